"""What each of the split path's products is worth (csrc/conv_split.hip).

Operands in neighbouring pairs (v, -bf16(v)) against equal ones: the leading
parts cancel, to zero and inside one matrix instruction, and what is left is
the product of v's lower parts, about 2^-10.3 of |v w| (a bf16 rounding is
uniform within 2^-9).  The products the kernels leave out (ml', lm', ll') are
within 2^-26 of |v w| together, so 2^-15.7 of the result; the small sums' own
roundings less.  A missing mm' is 2^-10.3 of it, a missing hl' or lh' about
2^-9.3, a missing hm' or mh' all.  The line is drawn at 2^-14."""
import math

import pytest
import torch
import torch.nn.functional as F

TERMS = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]   # of the first and the second operand: h, m, l
LINE = 2.0 ** -14


def _split(v):
    h = v.bfloat16().float()
    m = (v - h).bfloat16().float()
    return h, m, (v - h - m).bfloat16().float()


def _paired(shape, dim, cancels, g, first=0):
    """Values in pairs along dim: (v, -bf16(v)) or (v, v); first: the index of
    the first pair (the ones before and a single one behind are 0)."""
    n = shape[dim] - first
    half = [*shape]
    half[dim] = n // 2
    v = torch.randn(half, generator=g)
    w = -v.bfloat16().float() if cancels else v
    body = torch.stack((v, w), dim + 1).flatten(dim, dim + 1)
    pad = [0, 0] * len(shape)
    pad[2 * (len(shape) - 1 - dim)] = first
    pad[2 * (len(shape) - 1 - dim) + 1] = n % 2
    return F.pad(body, pad)


def _conv_operands(which, cin=64, cout=72, h=20, w=36):
    g = torch.Generator().manual_seed(cin + (which == "weight"))
    return (_paired((1, cin, h, w), 1, which == "input", g),
            _paired((cout, cin, 3, 3), 1, which == "weight", g))


def _wgrad_operands(which, first, cin=64, cout=70, h=90, w=48):
    """The pairs along the columns; the gradient's start at `first`."""
    g = torch.Generator().manual_seed(first + (which == "gradient"))
    return _paired((1, cin, h, w), 3, which == "input", g), _paired((1, cout, h, w), 3, which == "gradient", g, first)


def _wgrad(x, gz, first):
    """The weight gradient's taps whose products stay in pairs: the middle
    column for gradients that start at 0, the two others at 1."""
    h, w = x.shape[2:]
    cols = (0, 2) if first else (1,)
    xp, z = F.pad(x[0], (1, 1, 1, 1)), gz[0].flatten(1)
    return torch.stack([z @ xp[:, a:a + h, b:b + w].flatten(1).t().contiguous() for a in range(3) for b in cols], -1)


def _error(y, y64):
    return float((y.double() - y64).norm() / y64.norm())


def _sum_of(products, f, a, b):
    a, b = _split(a), _split(b)
    return sum(f(a[i].double(), b[j].double()) for i, j in products)


CASES = [("conv", "input", 0), ("conv", "weight", 0), ("wgrad", "input", 0), ("wgrad", "input", 1),
         ("wgrad", "gradient", 0), ("wgrad", "gradient", 1)]


@pytest.mark.parametrize("kind,which,first", CASES)
def test_the_line_lies_between_six_products_and_five(kind, which, first):
    """On the CPU, products added in 64 bits: all six within the line.  Without
    one of the small ones beyond it, in the case whose pairs leave it in (the l
    part of the operand that cancels)."""
    if kind == "conv":
        a, b = _conv_operands(which)
        f = lambda x, w: F.conv2d(x, w, padding=1)                        # noqa: E731
    else:
        a, b = _wgrad_operands(which, first)
        f = lambda x, z: _wgrad(x, z, first)                              # noqa: E731
    want = f(a.double(), b.double())
    assert _error(_sum_of(TERMS, f, a, b), want) <= LINE / 2
    kept = (2, 0) if which == "input" else (0, 2)
    lost = (1, 0) if which == "input" else (0, 1)
    for term in ((1, 1), kept, lost):
        assert _error(_sum_of([t for t in TERMS if t != term], f, a, b), want) >= 4 * LINE, term


@pytest.mark.gpu
@pytest.mark.parametrize("kind,which,first", CASES)
def test_every_product_counts(pkg, kind, which, first):
    from tests.test_conv_split import _split_conv
    C = pkg.convnet
    if kind == "conv":
        x, wt = (t.cuda() for t in _conv_operands(which))
        want = F.conv2d(x.double(), wt.double(), padding=1)
        assert _error(_split_conv(pkg, x, C.pack3x3(wt), wt.shape[0]), want) <= LINE
        gate = torch.ones_like(x)
        assert _error(_split_conv(pkg, x, C.pack3x3(wt), wt.shape[0], act="relu", gate=gate), want) <= LINE
        return
    x, gz = (t.cuda() for t in _wgrad_operands(which, first))
    n, cin, h, w = x.shape
    assert 18 * n * cin * gz.shape[1] * h * w >= 1.5e8 and w >= 16
    gw = C.conv3x3_wgrad(x, gz, gz.shape[1])
    cols = (0, 2) if first else (1,)
    got = torch.stack([gw[:, :, a, b] for a in range(3) for b in cols], -1)
    assert _error(got, _wgrad(x.double(), gz.double(), first)) <= LINE


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 128, 256, 128, 128), (9, 64, 64, 96, 96), (1, 512, 512, 32, 32),
                                   (4, 512, 512, 16, 16)])
def test_error_and_bias_of_large_layers(pkg, shape):
    """Unsplit and in K slices.  Norm-wise: the sum is truncated once per 16
    products, 2^-24 of it on average and with alternating sign, so sqrt(9 Cin /
    16) of that, and 2^-23 for the rest.  The mean error is below 1e-9 of the
    products' magnitudes (3e-9 at 128 channels without the change of sign)."""
    n, cin, cout, h, w = shape
    C = pkg.convnet
    assert pkg._lib.query("svbrdf_conv3x3_split_preferred", n, cin, h, w, cout)
    g = torch.Generator().manual_seed(cin)
    x, wt = torch.randn((n, cin, h, w), generator=g).cuda(), (torch.randn((cout, cin, 3, 3), generator=g)
                                                              / math.sqrt(9 * cin)).cuda()
    bound = math.sqrt(9 * cin / 16) * 2.0 ** -24 + 2.0 ** -23
    with torch.no_grad():
        y = C.conv3x3(x, wt).double()
    want = F.conv2d(x.double(), wt.double(), padding=1)
    size = F.conv2d(x.double().abs(), wt.double().abs(), padding=1)
    assert _error(y, want) <= bound
    assert abs(float((y - want).mean() / size.mean())) <= 1e-9
    if n == 1:
        gz = torch.randn((n, cout, h, w), generator=g).cuda()
        gw = C.conv3x3_wgrad(x, gz, cout).double()
        xp, z = F.pad(x[0].double(), (1, 1, 1, 1)), gz[0].double().flatten(1)
        mid = z @ xp[:, 1:1 + h, 1:1 + w].flatten(1).t().contiguous()
        size = z.abs() @ xp[:, 1:1 + h, 1:1 + w].abs().flatten(1).t().contiguous()
        assert _error(gw[:, :, 1, 1], mid) <= math.sqrt(h * w / 16) * 2.0 ** -24 + 2.0 ** -23
        assert abs(float((gw[:, :, 1, 1] - mid).mean() / size.mean())) <= 1e-9
