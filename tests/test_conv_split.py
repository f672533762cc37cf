"""The 3x3 convolution on the bf16 matrix cores with split fp32 operands
(csrc/conv_split.hip) against the fp32 kernel and torch's FP64 convolution.

Bound of an output's error, relative to the convolution of |x| with |w|: one
truncation of the running sum per 16 products (2^-23 each: 9 Cin / 16 of
them), the five small product sums' truncations at 2^-8 of that (5 x 2^-8 <
1/32 more), the dropped products (3 x 2^-25) and the roundings of the split,
the slices' sum and the epilogue (16 x 2^-23 covers them)."""
import ctypes
import math

import pytest
import torch
import torch.nn.functional as F

from tests import convnet_ref as R

DEV = "cuda:0"


def _fake(i=1):
    return ctypes.c_void_p(0x10000 * i)


def test_split_entry_points_refuse_on_the_host(pkg):
    """Null pointers, fewer than 16 input channels, misaligned weights, an
    unknown activation and a short workspace are refused before any launch."""
    lib, f = pkg._lib.load(), _fake()
    assert lib.svbrdf_conv3x3_split_weights_bytes(0, 64) == 0
    # [chunks of 16][9 taps][3 terms][32-channel groups][1 KB], plus the factors
    assert lib.svbrdf_conv3x3_split_weights_bytes(33, 65) == 3 * 9 * 3 * 4 * 1024 + 65 * 4
    assert lib.svbrdf_conv3x3_pack_split(None, 64, 64, None, 1.0, 0, 0, f, None) == -1
    assert lib.svbrdf_conv3x3_pack_split(f, 64, 8, None, 1.0, 0, 0, f, None) == -2
    assert lib.svbrdf_conv3x3_pack_split(f, 8, 64, None, 1.0, 0, 1, f, None) == -2
    assert lib.svbrdf_conv3x3_pack_split(f, 64, 64, None, 1.0, 0, 0, ctypes.c_void_p(0x10008), None) == -1
    assert lib.svbrdf_conv3x3_split_packed(f, 15, 64, f, None) == -2
    assert lib.svbrdf_conv3x3_split_packed(f, 64, 64, None, None) == -1
    need = lib.svbrdf_conv3x3_split_workspace_bytes(1, 512, 16, 16, 512)
    assert need > 0 and need % (512 * 256 * 4) == 0
    assert lib.svbrdf_conv3x3_split_workspace_bytes(1, 15, 16, 16, 512) == 0
    assert lib.svbrdf_conv3x3_split(f, 1, 512, 16, 16, f, 512, None, None, 0.0, 0, f, f, need - 4, None) == -3
    assert lib.svbrdf_conv3x3_split(f, 1, 8, 16, 16, f, 512, None, None, 0.0, 0, f, None, 0, None) == -2
    assert lib.svbrdf_conv3x3_split(f, 1, 64, 16, 16, f, 64, None, None, 0.0, 7, f, f, 1 << 30, None) == -1
    assert lib.svbrdf_conv3x3_input_grad_split(f, None, 1, 1, 64, 16, 16, f, 64, f, None, 0, None) == -1
    assert lib.svbrdf_conv3x3_input_grad_split(f, f, 9, 1, 64, 16, 16, f, 64, f, None, 0, None) == -1


def test_split_rule(pkg):
    """The path is taken for large layers only: 2 GFLOP, 32 input channels,
    more than 8 output channels."""
    q = pkg._lib.load().svbrdf_conv3x3_split_preferred
    assert q(9, 64, 256, 256, 64) == 1 and q(1, 512, 32, 32, 512) == 1
    assert q(9, 3, 256, 256, 64) == 0 and q(9, 31, 256, 256, 64) == 0 and q(9, 64, 256, 256, 8) == 0
    assert q(1, 512, 16, 16, 512) == 0 and q(0, 64, 256, 256, 64) == 0


def _layer(shape, seed):
    n, cin, cout, h, w = shape
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((n, cin, h, w), generator=g)
    wt = torch.randn((cout, cin, 3, 3), generator=g) / math.sqrt(9 * cin)
    return x.to(DEV), wt.to(DEV), (0.1 * torch.randn(cout, generator=g)).to(DEV), torch.randn((1, 1, h, w), generator=g).to(DEV)


def _split_conv(pkg, x, packed, cout, bias=None, noise=None, strength=0.0, act="none", gate=None):
    """The split entry points at any shape (convnet takes them by its rule)."""
    from svbrdf_amd import _lib, convnet
    n, cin, h, w = x.shape
    split = convnet._split_packed(packed)
    y = torch.empty((n, cout, h, w), device=DEV)
    nb = _lib.query("svbrdf_conv3x3_split_workspace_bytes", n, cin, h, w, cout)
    ws = torch.empty(nb // 4 + 1, device=DEV)
    s = _lib.stream_handle(x.device)
    if gate is None:
        _lib.call("svbrdf_conv3x3_split", _lib.ptr(x), n, cin, h, w, _lib.ptr(split), cout, _lib.ptr(bias),
                  _lib.ptr(noise), strength, convnet.ACT[act], _lib.ptr(y), _lib.ptr(ws), nb, s)
    else:
        _lib.call("svbrdf_conv3x3_input_grad_split", _lib.ptr(x), _lib.ptr(gate), convnet.ACT[act], n, cin, h, w,
                  _lib.ptr(split), cout, _lib.ptr(y), _lib.ptr(ws), nb, s)
    return y


def _bound(cin):
    return (9 * cin / 16 * (1 + 1 / 32) + 16) * 2.0 ** -23


# n, cin, cout, h, w: tile edges (128- and 256-pixel tiles of 4 to 32 columns),
# 64- and 128-channel blocks with remainders, partial last chunks, K slices
SHAPES = [(1, 16, 9, 1, 1), (2, 64, 64, 37, 29), (1, 17, 70, 5, 7), (3, 128, 256, 24, 40), (1, 512, 512, 4, 4),
          (1, 512, 130, 16, 16), (2, 33, 36, 17, 300), (1, 40, 200, 3, 50), (1, 95, 65, 70, 3), (9, 64, 64, 9, 33),
          (1, 48, 128, 256, 256)]


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["none", "relu", "lrelu"])
@pytest.mark.parametrize("shape", SHAPES, ids=[f"{s[0]}x{s[1]}->{s[2]}@{s[3]}x{s[4]}" for s in SHAPES])
def test_split_conv_against_fp64(pkg, shape, act):
    """Forward with every epilogue, and the gated input gradient's
    convolution, within the derived bound; the same bits on every run."""
    from svbrdf_amd import convnet
    n, cin, cout, h, w = shape
    x, wt, b, nz = _layer(shape, sum(shape))
    packed = convnet.pack3x3(wt)
    y = _split_conv(pkg, x, packed, cout, b, nz, 0.37, act)
    assert torch.equal(y, _split_conv(pkg, x, packed, cout, b, nz, 0.37, act))
    y64 = R.conv3x3_ref(x.double(), wt.double(), b, nz, 0.37, act)
    scale = F.conv2d(x.double().abs(), wt.double().abs(), padding=1) + 0.37 * nz.double().abs()
    scale = (scale + b.double().abs().view(1, -1, 1, 1)) * math.sqrt(2.0)
    worst = float(((y.double() - y64).abs() / (_bound(cin) * scale)).max())
    assert worst <= 1.0, worst
    gate = torch.randn(x.shape, generator=torch.Generator().manual_seed(1)).to(DEV)
    slope = {"none": (1.0, 1.0), "relu": (1.0, 0.0), "lrelu": (math.sqrt(2.0), 0.2 * math.sqrt(2.0))}[act]
    gated = x.double() * torch.where(gate > 0, slope[0], slope[1])
    g = _split_conv(pkg, x, packed, cout, act=act, gate=gate)
    scale = F.conv2d(gated.abs(), wt.double().abs(), padding=1)
    worst = float(((g.double() - F.conv2d(gated, wt.double(), padding=1)).abs() / (_bound(cin) * scale + 1e-30)).max())
    assert worst <= 1.0, worst


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 48, 40), (1, 33, 70), (1, 130, 64)])
@pytest.mark.parametrize("transpose", [False, True])
def test_split_packing_is_the_packed_weights(pkg, shape, transpose):
    """Modulated, demodulated weights packed straight into the split layout
    are the bits that splitting pack3x3's output gives, and every value is the
    sum of its three terms."""
    from svbrdf_amd import _lib, convnet
    _, cin, cout = shape
    g = torch.Generator().manual_seed(cin)
    wt, style = torch.randn((cout, cin, 3, 3), generator=g).to(DEV), (torch.rand(cin, generator=g) + 0.5).to(DEV)
    packed = convnet.pack3x3(wt, style, 0.07, True, transpose)
    a = convnet._split_packed(packed)
    b = torch.zeros_like(a)
    _lib.call("svbrdf_conv3x3_pack_split", _lib.ptr(wt), cout, cin, _lib.ptr(style), 0.07, 1, int(transpose), _lib.ptr(b),
              _lib.stream_handle(wt.device))
    k, m = packed.shape[1:]
    chunks, groups = (k + 15) // 16, (m + 63) // 64 * 2
    used = chunks * 9 * 3 * groups * 64 * 4
    assert torch.equal(a[:used].view(torch.int32), b[:used].view(torch.int32))
    # [chunk, tap, term, group, half, row, 8] of bf16
    terms = a[:used].view(torch.bfloat16).double().view(chunks, 9, 3, groups, 2, 32, 8)
    val = terms.sum(2).permute(1, 0, 3, 5, 2, 4)                  # tap, chunk, half, 8, group, row
    val = val.reshape(9, chunks, 16, groups * 32)[..., :m]
    val = val * torch.tensor([(-1.0) ** c for c in range(chunks)], device=DEV, dtype=torch.float64).view(1, -1, 1, 1)
    for c in range(chunks):
        lo = min(c * 16, k - 16)
        want = packed[:, lo:lo + 16].double().clone()
        want[:, : c * 16 - lo] = 0.0
        assert torch.equal(val[:, c], want)


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["input", "weight", "both", "large"])
def test_split_conv_spreads_infinities_like_fp32(pkg, where):
    """Infinities, NaN and values that round to infinity in bf16, in the input
    or the weights: the outputs they reach are the fp32 kernel's (same NaN and
    signed infinities), and the others are finite and close."""
    from svbrdf_amd import _lib, convnet
    n, cin, cout, h, w = 1, 40, 72, 20, 36
    x, wt, _, _ = _layer((n, cin, cout, h, w), 7)
    if where in ("input", "both"):
        x[0, 3, 5, 6], x[0, 33, 15, 30], x[0, 20, 0, 0] = float("inf"), float("nan"), float("-inf")
    if where in ("weight", "both"):
        wt[9, 4, 1, 1], wt[65, 39, 0, 2] = float("-inf"), float("nan")
    if where == "large":
        x[0, 3, 5, 6], x[0, 39, 11, 11] = 3.4e38, -3.4e38
        wt[7, 11, 0, 0] = 3.4e38
        wt *= 2.0 ** -12      # the sums themselves stay finite but for that weight's
        wt[7, 11, 0, 0] = 3.4e38
    packed = convnet.pack3x3(wt)
    y = _split_conv(pkg, x, packed, cout)
    ref = torch.empty_like(y)
    nb = _lib.query("svbrdf_conv3x3_workspace_bytes", n, cin, h, w, cout)
    ws = torch.empty(nb // 4 + 1, device=DEV)
    _lib.call("svbrdf_conv3x3", _lib.ptr(x), n, cin, h, w, _lib.ptr(packed), cout, None, None, 0.0, 0, _lib.ptr(ref),
              _lib.ptr(ws), nb, _lib.stream_handle(x.device))
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isinf(y), torch.isinf(ref)) and torch.equal(y[torch.isinf(y)], ref[torch.isinf(ref)])
    ok = torch.isfinite(ref)
    scale = F.conv2d(x.double().abs().nan_to_num(0.0, 0.0, 0.0), wt.double().abs().nan_to_num(0.0, 0.0, 0.0), padding=1)
    # both sides' roundings: fp32's once per product pair
    bound = (_bound(cin) + 9 * cin / 2 * 2.0 ** -23) * scale + 1e-30
    assert bool(((y.double() - ref.double()).abs()[ok] <= bound[ok]).all())


# n, cin, cout, h, w: channel tiles with remainders, strips of 32 columns with
# remainders (vector rows and odd ones), strips that end inside a slice, slices
# that start inside a strip, one-row images, a single slice
WGRAD = [(1, 64, 64, 80, 32), (1, 70, 33, 90, 47), (2, 40, 130, 19, 45), (3, 65, 64, 9, 100), (1, 96, 200, 1, 700),
         (1, 512, 512, 16, 16), (9, 16, 16, 64, 64), (1, 130, 128, 60, 20)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", WGRAD, ids=[f"{s[0]}x{s[1]}->{s[2]}@{s[3]}x{s[4]}" for s in WGRAD])
def test_wgrad_split_against_fp64(pkg, shape):
    """The weight gradient on split operands: one truncation of the running
    sum per 16 pixels and those of the small sums, the slices' additions and the
    split's roundings, relative to the sum of |x| |dL/dz|; the same bits twice."""
    from svbrdf_amd import convnet
    n, cin, cout, h, w = shape
    assert w >= 16 and 18 * n * cin * cout * h * w >= 1.5e8        # the path under test
    g = torch.Generator().manual_seed(sum(shape))
    x, gz = torch.randn((n, cin, h, w), generator=g).to(DEV), torch.randn((n, cout, h, w), generator=g).to(DEV)
    gw = convnet.conv3x3_wgrad(x, gz, cout)
    assert torch.equal(gw, convnet.conv3x3_wgrad(x, gz, cout))

    def exact(x, gz):
        xp, z = F.pad(x.double(), (1, 1, 1, 1)), gz.double().transpose(0, 1).flatten(1)
        taps = [z @ xp[:, :, a:a + h, b:b + w].transpose(0, 1).flatten(1).t().contiguous()
                for a in range(3) for b in range(3)]
        return torch.stack(taps, -1).view(cout, cin, 3, 3)

    chunks = n * h * ((w + 31) // 32)
    bound = (2 * chunks * (1 + 1 / 32) + 256 + 16) * 2.0 ** -23 * exact(x.abs(), gz.abs())
    err = (gw.double() - exact(x, gz)).abs()        # a tap that meets no input row is 0 within 0
    assert bool((err <= bound).all()), float((err / (bound + 1e-300)).max())


@pytest.mark.gpu
def test_wgrad_split_spreads_infinities_like_fp32(pkg):
    """Non-finite inputs and gradients: the same NaN and signed infinities as a
    plain convolution's weight gradient in FP64 has, the rest finite."""
    from svbrdf_amd import convnet
    x, _, _, _ = _layer((1, 48, 8, 40, 64), 3)
    gz = torch.randn((1, 80, 40, 64), generator=torch.Generator().manual_seed(4)).to(DEV)
    x[0, 5, 20, 30], x[0, 40, 39, 63], x[0, 47, 10, 33] = float("inf"), float("nan"), -3.4e38
    gz[0, 70, 7, 8] = float("-inf")
    gz[0, :, 9:12, 32:35] *= 2.0 ** -10       # around the large value: finite products
    gw = convnet.conv3x3_wgrad(x, gz, 80)
    xp, z = F.pad(x.double(), (1, 1, 1, 1)), gz.double()[0].flatten(1)
    want = torch.stack([(z[:, None] * xp[0, :, a:a + 40, b:b + 64].flatten(1)[None]).sum(-1)
                        for a in range(3) for b in range(3)], -1).view(80, 48, 3, 3)
    assert torch.equal(torch.isnan(gw), torch.isnan(want))
    assert torch.equal(torch.isinf(gw), torch.isinf(want)) and torch.equal(gw[torch.isinf(gw)].double(), want[torch.isinf(want)])
