"""A convolution's second, scaled copy of its output on every kernel that
writes one, and the feature vector made of them: the same bits as the product
and the concatenation."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# at most 4 input channels; at most 8 output channels; the staged fp32 kernel,
# whole and K-split; the split-operand kernel, whole and K-split, both tiles
@pytest.mark.parametrize("n,cin,cout,h,w", [(2, 3, 70, 9, 13), (1, 64, 3, 33, 31), (1, 20, 24, 17, 19),
                                            (1, 512, 64, 8, 8), (4, 64, 64, 128, 97), (1, 512, 512, 32, 32),
                                            (3, 128, 128, 64, 66)])
@pytest.mark.parametrize("act", ["none", "relu", "lrelu"])
@pytest.mark.parametrize("offset", [0, 1])
def test_the_copy_is_the_scaled_output(pkg, n, cin, cout, h, w, act, offset):
    g = torch.Generator().manual_seed(3)
    layer = pkg.convnet.Conv3x3(torch.randn((cout, cin, 3, 3), generator=g).to(DEV) / (9 * cin) ** 0.5,
                                torch.randn(cout, generator=g).to(DEV), act=act)
    x = torch.randn((n, cin, h, w), generator=g).to(DEV)
    room = torch.full((n * cout * h * w + 8,), 7.0, device=DEV)
    tap = room[offset:offset + n * cout * h * w]
    y = layer(x, tap, 0.3)
    assert torch.equal(y, layer(x))
    assert torch.equal(tap.view_as(y), y * 0.3)
    rest = torch.cat([room[:offset], room[offset + tap.numel():]])
    assert bool((rest == 7.0).all())


@pytest.mark.parametrize("weights", [[1, 1, 4, 8], [0, 3, 1], [2]])
@pytest.mark.parametrize("n,h,w", [(1, 32, 32), (2, 37, 50)])
def test_the_feature_vector(pkg, weights, n, h, w):
    net = pkg.materialgan.VGGLoss(DEV, np.array(weights) / 14)
    x = torch.rand((n, 3, h, w), generator=torch.Generator().manual_seed(1)).to(DEV)
    got = net.compute_feature_vector(x)
    x.requires_grad_(True)
    ref = net.compute_feature_vector(x)
    assert ref.requires_grad and not got.requires_grad and torch.equal(got, ref.detach())
    with torch.no_grad():
        assert torch.equal(net.compute_feature_vector(x), ref)
    net.load(x)
    assert torch.equal(net.im_feature, net.compute_feature_vector(net.normalize(x)).detach())


def test_a_copy_is_refused_where_a_gradient_is_asked_for(pkg):
    layer = pkg.convnet.Conv3x3(torch.randn(16, 16, 3, 3, device=DEV))
    x, tap = torch.randn(1, 16, 4, 4, device=DEV), torch.empty(256, device=DEV)
    for bad in (torch.empty(255, device=DEV), torch.empty(512, device=DEV)[::2], torch.empty(256)):
        with pytest.raises(ValueError):
            layer(x, bad, 1.0)
    with pytest.raises(ValueError):
        layer(x.requires_grad_(True), tap, 1.0)
