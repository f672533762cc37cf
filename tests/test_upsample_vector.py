"""The row kernels of the generator's x2 upsampling and its adjoint, and the
vector form of the K slices' sum, at the edges of their rules: widths down to
one vector, remainders of the row strips, odd sizes and misaligned tensors,
which take the one-value kernels.

An output of the upsampling is four products with weights that are powers of
two or three quarters, summed in three additions, an input's gradient 16 in
15: within 4 and 16 roundings (2^-24 each) of the sum of |weight x value|."""
import pytest
import torch
import torch.nn.functional as F

from tests import convnet_ref as R

DEV = "cuda:0"


def _offset(shape, floats):
    """A tensor whose first value lies `floats` past a 256-byte boundary."""
    n = int(torch.Size(shape).numel())
    return torch.empty(n + 64, device=DEV)[floats:floats + n].view(shape)


# planes, h, w: both sides of the 2^18-value line, strips with a remainder
@pytest.mark.gpu
@pytest.mark.parametrize("planes,h,w", [(512, 4, 4), (512, 16, 16), (300, 33, 34), (40, 65, 31), (9000, 5, 2),
                                        (7, 97, 100), (3, 128, 256), (70, 1, 1024)])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_upsample_and_adjoint(pkg, planes, h, w, shift):
    from svbrdf_amd import _lib
    g = torch.Generator().manual_seed(planes + h + w)
    x, gy = _offset((1, planes, h, w), shift), _offset((1, planes, 2 * h, 2 * w), shift)
    x.copy_(torch.randn(x.shape, generator=g))
    gy.copy_(torch.randn(gy.shape, generator=g))
    y, gx, s = torch.empty_like(gy.contiguous()), torch.empty_like(x.contiguous()), _lib.stream_handle(x.device)
    out = [_offset(t.shape, shift) for t in (y, gx)]
    _lib.call("svbrdf_upsample2_blur", _lib.ptr(x), planes, h, w, _lib.ptr(out[0]), s)
    _lib.call("svbrdf_upsample2_blur_adjoint", _lib.ptr(gy), planes, h, w, _lib.ptr(out[1]), s)
    x64 = x.double().requires_grad_(True)
    y64 = R.upsample2_ref(x64)
    (g64,) = torch.autograd.grad(y64, x64, gy.double())
    a64 = x.double().abs().requires_grad_(True)
    s64 = R.upsample2_ref(a64)
    (t64,) = torch.autograd.grad(s64, a64, gy.double().abs())
    assert bool(((out[0].double() - y64).abs() <= 4 * 2.0 ** -24 * s64 + 1e-30).all())
    assert bool(((out[1].double() - g64).abs() <= 16 * 2.0 ** -24 * t64 + 1e-30).all())


@pytest.mark.gpu
@pytest.mark.parametrize("side,shift", [(4, 0), (4, 1), (5, 0), (6, 2)])
def test_slice_sum_epilogue(pkg, side, shift):
    """A K-split layer with noise, bias and leaky ReLU, whose slices are summed
    four pixels at a time (side^2 a multiple of 4, aligned output) or one:
    within 2e-5 of FP64 relative to the convolution of |x| with |w|, and the
    vector form has the bits of the other."""
    from svbrdf_amd import _lib, convnet
    n, cin, cout = 2, 512, 96
    g = torch.Generator().manual_seed(side)
    x, wt = torch.randn((n, cin, side, side), generator=g).to(DEV), torch.randn((cout, cin, 3, 3), generator=g).to(DEV)
    b, nz = torch.randn(cout, generator=g).to(DEV), torch.randn((1, 1, side, side), generator=g).to(DEV)
    packed = convnet.pack3x3(wt)
    nb = _lib.query("svbrdf_conv3x3_workspace_bytes", n, cin, side, side, cout)
    assert nb >= 2 * n * cout * side * side * 4
    ws, s = torch.empty(nb // 4, device=DEV), _lib.stream_handle(x.device)

    def conv(y):
        _lib.call("svbrdf_conv3x3", _lib.ptr(x), n, cin, side, side, _lib.ptr(packed), cout, _lib.ptr(b), _lib.ptr(nz),
                  0.3, convnet.ACT["lrelu"], _lib.ptr(y), _lib.ptr(ws), nb, s)
        return y

    y = conv(_offset((n, cout, side, side), shift))
    assert torch.equal(y, conv(_offset((n, cout, side, side), 1)))
    y64 = R.conv3x3_ref(x.double(), wt.double(), b, nz, 0.3, "lrelu")
    scale = F.conv2d(x.double().abs(), wt.double().abs(), padding=1)
    assert bool(((y.double() - y64).abs() <= 2e-5 * scale + 1e-7).all())
