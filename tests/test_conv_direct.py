"""The convolution to at most eight output channels: both ways its weights
travel, chunks of eight channels with a remainder, blocks that hang over the
image's edges, and its gated form.

Tolerance, per value: K = 9 Cin products and their sum, each off by at most
2^-24 of the running sum of magnitudes, and the gate's product."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("cout", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("n,cin,h,w", [(1, 1, 1, 1), (2, 8, 8, 64), (1, 9, 9, 65), (3, 23, 17, 130), (1, 64, 40, 33)])
def test_against_float64(pkg, n, cin, cout, h, w):
    C, g = pkg.convnet, torch.Generator().manual_seed(8)
    x, y = torch.randn((n, cin, h, w), generator=g), torch.randn((n, cin, h, w), generator=g)
    wt = torch.randn((cout, cin, 3, 3), generator=g)
    packed = C.pack3x3(wt.to(DEV))
    gate = torch.where(y > 0, 1.0, 0.2).double() * 2 ** 0.5
    for got, inp in ((C.conv3x3_packed(x.to(DEV), packed, cout), x.double()),
                     (C.conv3x3_input_grad(x.to(DEV), y.to(DEV), packed, cout, "lrelu"), x.double() * gate)):
        ref = F.conv2d(inp, wt.double(), padding=1)
        size = F.conv2d(inp.abs(), wt.double().abs(), padding=1)
        assert bool(((got.cpu().double() - ref).abs() <= (9 * cin + 4) * 2.0 ** -24 * size).all())
