"""The 3x3 convolution of at most four input channels: odd and small images,
ragged channel counts, every epilogue, and the gated input gradient.

Tolerance, per value: K = 9 Cin products and at most three more operations in
fp32, each off by at most 2^-24 of the running sum of magnitudes, times the
activation's sqrt(2): 1.5 (K + 4) 2^-24 sum(|x| |w|, |noise|, |bias|)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ACT = {"none": lambda v: v, "relu": torch.relu, "lrelu": lambda v: F.leaky_relu(v, 0.2) * 2 ** 0.5}


@pytest.mark.parametrize("act", ["none", "relu", "lrelu"])
@pytest.mark.parametrize("n,cin,cout,h,w", [(1, 1, 9, 1, 1), (2, 3, 64, 5, 7), (1, 2, 65, 33, 1), (3, 4, 130, 8, 32),
                                            (1, 3, 63, 100, 101), (1, 4, 12, 1, 300), (9, 3, 64, 130, 66)])
def test_against_float64(pkg, n, cin, cout, h, w, act):
    C, g = pkg.convnet, torch.Generator().manual_seed(5)
    x, wt = torch.randn((n, cin, h, w), generator=g), torch.randn((cout, cin, 3, 3), generator=g)
    bias, noise = torch.randn(cout, generator=g), torch.randn(h, w, generator=g)
    packed = C.pack3x3(wt.to(DEV))
    y = C.conv3x3_packed(x.to(DEV), packed, cout, bias.to(DEV), noise.to(DEV), 0.5, act).cpu().double()
    conv = lambda a, b: F.conv2d(a.double(), b.double(), padding=1)   # noqa: E731
    ref = ACT[act](conv(x, wt) + 0.5 * noise.double() + bias.double().view(-1, 1, 1))
    size = conv(x.abs(), wt.abs()) + 0.5 * noise.double().abs() + bias.double().abs().view(-1, 1, 1)
    assert bool(((y - ref).abs() <= 1.5 * (9 * cin + 4) * 2.0 ** -24 * size).all())

    # the input gradient of a layer with cin output channels (gated input)
    if act == "none" or cout <= 8:
        return
    fwd = ACT[act](torch.randn((n, cin, h, w), generator=g))
    gate = torch.where(fwd > 0, 1.0, 0.0 if act == "relu" else 0.2) * (1.0 if act == "relu" else 2 ** 0.5)
    gx = C.conv3x3_input_grad(x.to(DEV), fwd.to(DEV), packed, cout, act).cpu().double()
    gated = x.double() * gate.double()
    assert bool(((gx - conv(gated, wt)).abs() <= 1.5 * (9 * cin + 4) * 2.0 ** -24 * conv(gated.abs(), wt.abs())).all())


@pytest.mark.parametrize("cin", [1, 3])
def test_an_infinite_pixel_stays_where_it_is(pkg, cin):
    # an odd K: the padding product of the last step is zero whatever x holds
    x, wt = torch.ones((1, cin, 12, 12), device=DEV), torch.ones((16, cin, 3, 3), device=DEV)
    x[0, cin - 1, 5, 5] = float("inf")
    y = pkg.convnet.conv3x3_packed(x, pkg.convnet.pack3x3(wt), 16)
    seen = torch.zeros((12, 12), dtype=torch.bool, device=DEV)
    seen[4:7, 4:7] = True
    assert bool((torch.isinf(y[0]) == seen).all()) and not bool(torch.isnan(y).any())
