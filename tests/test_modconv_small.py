"""The modulated convolution of at most 128 pixels from the network's own
weights: every split of waves and pixels, odd images, ragged channel counts.

Tolerance, per value: an accumulator takes at most 4 rounds of 36 steps of two
products, the slices' and waves' sums fewer than 32 more, the weights, the
demodulation factor and the epilogue under 50 roundings: 400 of 2^-24 of the
sum of magnitudes, times the activation's sqrt(2)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ACT = {"none": lambda v: v, "relu": torch.relu, "lrelu": lambda v: F.leaky_relu(v, 0.2) * 2 ** 0.5}


@pytest.mark.parametrize("demodulate", [True, False])
@pytest.mark.parametrize("cin,cout,h,w,act", [
    (512, 512, 4, 4, "lrelu"), (8, 1, 1, 1, "none"), (40, 33, 5, 7, "relu"), (512, 64, 8, 8, "lrelu"),
    (96, 70, 1, 64, "none"), (64, 96, 13, 5, "lrelu"), (72, 40, 10, 11, "relu"), (512, 512, 8, 16, "lrelu"),
    (24, 65, 1, 128, "none"), (256, 31, 128, 1, "lrelu")])
def test_against_float64(pkg, cin, cout, h, w, act, demodulate):
    C, g = pkg.convnet, torch.Generator().manual_seed(11)
    assert int(pkg._lib.query("svbrdf_modconv3x3_small_workspace_bytes", cin, h, w, cout))
    x, wt = torch.randn((1, cin, h, w), generator=g), torch.randn((cout, cin, 3, 3), generator=g)
    style, bias = torch.randn(cin, generator=g), torch.randn(cout, generator=g)
    noise, scale = torch.randn(h, w, generator=g), (9 * cin) ** -0.5
    y = C.modulated_conv3x3(x.to(DEV), style.to(DEV), wt.to(DEV), scale, demodulate, bias.to(DEV), noise.to(DEV), 0.3,
                            act).cpu().double()
    w64 = wt.double() * scale * style.double().view(1, -1, 1, 1)
    if demodulate:
        w64 = w64 / (w64.pow(2).sum((1, 2, 3), keepdim=True) + 1e-8).sqrt()
    tail = 0.3 * noise.double() + bias.double().view(-1, 1, 1)
    ref = ACT[act](F.conv2d(x.double(), w64, padding=1) + tail)
    size = F.conv2d(x.double().abs(), w64.abs(), padding=1) + tail.abs()
    assert bool(((y - ref).abs() <= 1.5 * 400 * 2.0 ** -24 * size).all())


def test_the_shapes_that_pack(pkg):
    q = lambda *a: int(pkg._lib.query("svbrdf_modconv3x3_small_workspace_bytes", *a))   # noqa: E731
    assert q(512, 3, 43, 512) == 0 and q(20, 4, 4, 32) == 0 and q(0, 4, 4, 32) == 0
    # weights that are not 16-byte aligned take the packed path
    C, g = pkg.convnet, torch.Generator().manual_seed(2)
    room = torch.randn(16 * 16 * 9 + 1, generator=g).to(DEV)
    x, style = torch.randn((1, 16, 6, 6), generator=g).to(DEV), torch.randn(16, generator=g).to(DEV)
    odd = room[1:].view(16, 16, 3, 3)
    a = C.modulated_conv3x3(x, style, odd, 0.1, True)
    b = C.modulated_conv3x3(x, style, odd.clone(), 0.1, True)
    assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())
