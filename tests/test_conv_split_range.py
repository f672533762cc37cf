"""Small operands on the split path (csrc/conv_split.hip).

Below 2^-110 an fp32 value is no sum of three bf16 values: at 2^-122 the split
alone would be off by up to 2^-134 / 2^-122 = 2.4e-4.  Such operands, and sums
whose low products would leave fp32's range, go through the fp32 instruction.
Tolerance, norm-wise: that instruction rounds the sum once per product pair,
2^-24 each and of either sign, so four times sqrt(products / 2) of them."""
import math

import pytest
import torch
import torch.nn.functional as F

from tests.test_conv_split import _split_conv

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _values(shape, exponent, g):
    """Both signs, magnitudes in [1, 2) times 2^exponent: 24 bits each, no subnormals."""
    v = (1 + torch.rand(shape, generator=g)) * (torch.randint(0, 2, shape, generator=g) * 2 - 1)
    return (v * 2.0 ** exponent).to(DEV)


def _error(y, y64):
    return float((y.double() - y64).norm() / y64.norm())


# exponents of the input and the weights: either below the line, products and
# sums below it from operands above it, both above it and the sums as well
EXPONENTS = [(-122, 0), (0, -122), (-105, 0), (-60, -60), (-100, 0), (-98, 90)]


@pytest.mark.parametrize("xe,we", EXPONENTS)
@pytest.mark.parametrize("shape", [(1, 64, 72, 20, 36), (1, 200, 64, 9, 9)])
def test_convolution(pkg, shape, xe, we):
    """Forward and gated, unsplit and in K slices."""
    from svbrdf_amd import convnet
    n, cin, cout, h, w = shape
    g = torch.Generator().manual_seed(cin)
    x, wt = _values((n, cin, h, w), xe, g), _values((cout, cin, 3, 3), we, g)
    gate = torch.randn(x.shape, generator=g).to(DEV)
    tol = 4 * math.sqrt(9 * cin / 2) * 2.0 ** -24
    y = _split_conv(pkg, x, convnet.pack3x3(wt), cout)
    assert _error(y, F.conv2d(x.double(), wt.double(), padding=1)) <= tol
    y = _split_conv(pkg, x, convnet.pack3x3(wt), cout, act="relu", gate=gate)
    assert _error(y, F.conv2d(x.double() * (gate > 0), wt.double(), padding=1)) <= tol


def test_subnormal_terms(pkg):
    """Powers of two among the subnormal numbers: their first term is all of
    them, and it counts in either operand."""
    from svbrdf_amd import convnet
    cin, cout, h, w = 64, 70, 90, 47
    g = torch.Generator().manual_seed(6)

    def small(shape):
        e = torch.randint(-133, -125, shape, generator=g)
        return torch.ldexp((torch.randint(0, 2, shape, generator=g) * 2 - 1).double(), e).float().to(DEV)

    x, wt = small((1, cin, h, w)), _values((cout, cin, 3, 3), 60, g)
    tol = 4 * math.sqrt(9 * cin / 2) * 2.0 ** -24
    y = _split_conv(pkg, x, convnet.pack3x3(wt), cout)
    assert _error(y, F.conv2d(x.double(), wt.double(), padding=1)) <= tol
    gz = _values((1, cout, h, w), 60, g)
    tol = 4 * math.sqrt(h * w / 2) * 2.0 ** -24
    for a, b, rows in ((x, gz, cout), (gz, x, cin)):
        gw = convnet.conv3x3_wgrad(a, b, rows)
        mid = b[0].double().flatten(1) @ a[0].double().flatten(1).t().contiguous()
        assert _error(gw[:, :, 1, 1], mid) <= tol


@pytest.mark.parametrize("where", ["pixel", "channel", "weight", "row"])
def test_among_ordinary_values(pkg, where):
    """A pixel, an input channel, a weight or an output channel of small values
    among ordinary ones: the outputs that only those reach keep their bits."""
    from svbrdf_amd import convnet
    cin, cout, h, w = 48, 80, 24, 40
    g = torch.Generator().manual_seed(5)
    x, wt = _values((1, cin, h, w), 0, g), _values((cout, cin, 3, 3), -4, g)
    if where == "pixel":
        x[0, :, 4:9, 7:13] *= 2.0 ** -122
        rows, ys, xs = slice(0, cout), slice(5, 8), slice(8, 12)
    elif where == "channel":
        x[0, 20] *= 2.0 ** -122
        wt[33, :20], wt[33, 21:] = 0.0, 0.0
        rows, ys, xs = slice(33, 34), slice(0, h), slice(0, w)
    elif where == "weight":
        wt[70, 40, 1, 1] = -1.3 * 2.0 ** -120
        wt[70, :40], wt[70, 41:] = 0.0, 0.0
        wt[70, 40, 0], wt[70, 40, 2], wt[70, 40, 1, ::2] = 0.0, 0.0, 0.0
        rows, ys, xs = slice(70, 71), slice(0, h), slice(0, w)
    else:
        wt[9] *= 2.0 ** -118
        rows, ys, xs = slice(9, 10), slice(0, h), slice(0, w)
    y, y64 = _split_conv(pkg, x, convnet.pack3x3(wt), cout), F.conv2d(x.double(), wt.double(), padding=1)
    tol = 4 * math.sqrt(9 * cin / 2) * 2.0 ** -24
    assert _error(y[0, rows, ys, xs], y64[0, rows, ys, xs]) <= tol
    assert _error(y, y64) <= tol


@pytest.mark.parametrize("xe,ge", [(-122, 0), (0, -122), (-60, -60), (-105, 3)])
def test_weight_gradient(pkg, xe, ge):
    from svbrdf_amd import convnet
    n, cin, cout, h, w = 1, 64, 70, 90, 47
    assert 18 * n * cin * cout * h * w >= 1.5e8 and w >= 16        # the path under test
    g = torch.Generator().manual_seed(8)
    x, gz = _values((n, cin, h, w), xe, g), _values((n, cout, h, w), ge, g)

    def exact(x, gz):
        xp, z = F.pad(x[0].double(), (1, 1, 1, 1)), gz[0].double().flatten(1)
        taps = [z @ xp[:, a:a + h, b:b + w].flatten(1).t().contiguous() for a in range(3) for b in range(3)]
        return torch.stack(taps, -1).view(cout, cin, 3, 3)

    tol = 4 * math.sqrt(h * w / 2) * 2.0 ** -24
    assert _error(convnet.conv3x3_wgrad(x, gz, cout), exact(x, gz)) <= tol
    # one column of pixels at a strip's edge, another inside an octet, small among ordinary ones
    x, gz = _values((n, cin, h, w), 0, g), _values((n, cout, h, w), 0, g)
    x[0, 5] = 0.0
    x[0, 5, :, 31] = _values((h,), -122, g)
    x[0, 40] = 0.0
    x[0, 40, 17, 21] = 1.7 * 2.0 ** -120
    gz[0, 60] = 0.0
    gz[0, 60, :, 32] = _values((h,), -120, g)
    gw, want = convnet.conv3x3_wgrad(x, gz, cout), exact(x, gz)
    for got, ref in ((gw[:, 5], want[:, 5]), (gw[:, 40], want[:, 40]), (gw[60], want[60]), (gw, want)):
        assert _error(got, ref) <= tol
