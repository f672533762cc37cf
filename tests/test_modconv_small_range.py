"""The modulated convolution of a few pixels where the style is far from 1: the
demodulated output is an ordinary number, its undemodulated sum is not.

Tolerance, norm-wise: the same roundings as at ordinary values, fewer than 400
of 2^-24 per output; subnormal intermediate sums would be off by far more (at
2^-130 a sum has 19 bits, at 2^-140 nine) and overflowed ones are infinite."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("side", [4, 8, 11])
@pytest.mark.parametrize("style_size,x_size", [(2.0 ** 60, 2.0 ** 66), (2.0 ** 70, 1.0), (2.0 ** -30, 2.0 ** -100),
                                               (2.0 ** -9, 2.0 ** -118), (1.0, 1.0)])
def test_style_far_from_one(pkg, side, style_size, x_size):
    cin, cout = 64, 40
    g = torch.Generator().manual_seed(side)
    assert int(pkg._lib.query("svbrdf_modconv3x3_small_workspace_bytes", cin, side, side, cout))
    x = ((1 + torch.rand((1, cin, side, side), generator=g)) * x_size).to(DEV)
    style = ((1 + torch.rand(cin, generator=g)) * style_size).to(DEV)
    wt = torch.randn((cout, cin, 3, 3), generator=g).to(DEV)
    y = pkg.convnet.modulated_conv3x3(x, style, wt, 0.0416, True)
    squares = (wt.double() * float(torch.tensor(0.0416)) * style.double().view(1, -1, 1, 1)).pow(2).sum((1, 2, 3), keepdim=True)
    # a sum of squares beyond fp32 is infinite there, and the factor 0
    factor = torch.where(squares > 3.4e38, torch.zeros_like(squares), (squares + 1e-8).rsqrt())
    w64 = wt.double() * float(torch.tensor(0.0416)) * style.double().view(1, -1, 1, 1) * factor
    ref = F.conv2d(x.double(), w64, padding=1)
    assert bool(torch.isfinite(y).all())
    size = F.conv2d(x.double().abs(), w64.abs(), padding=1)
    assert bool(((y.double() - ref).abs() <= 400 * 2.0 ** -24 * size).all())
