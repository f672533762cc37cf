"""A frozen layer whose packed weights are replaced or written to after it was
built, or that was saved by a build without split weights."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _weights(cin, cout, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn((cout, cin, 3, 3), generator=g) / math.sqrt(9 * cin)).to(DEV)


@pytest.mark.parametrize("how", ["replaced", "written", "inference", "saved"])
def test_split_weights_follow_the_packed_ones(pkg, how):
    """Forward, input gradient and pooled output at a size of the split path are
    those of a layer built from the new weights, to the bit."""
    C = pkg.convnet
    cin, cout, n, side = 64, 64, 2, 160
    assert pkg._lib.query("svbrdf_conv3x3_split_preferred", n, cin, side, side, cout)
    old, new = _weights(cin, cout, 1), _weights(cin, cout, 2)
    fresh = C.Conv3x3(new)
    if how == "saved":
        layer = C.Conv3x3(new)
        for name in ("_splits", "split", "split_t"):
            layer.__dict__.pop(name, None)
    elif how == "written":
        layer = C.Conv3x3(old)
        layer.packed.copy_(fresh.packed)
        layer.packed_t.copy_(fresh.packed_t)
    else:
        with torch.inference_mode(how == "inference"):
            layer = C.Conv3x3(old)
            layer.packed, layer.packed_t = C.pack3x3(new), C.pack3x3(new, transpose=True)
    x = torch.randn((n, cin, side, side), generator=torch.Generator().manual_seed(3)).to(DEV)

    def passes(conv):
        leaf = x.clone().requires_grad_(True)
        y = conv(leaf)
        y.backward(torch.ones_like(y))
        with torch.no_grad():
            return y.detach(), leaf.grad, conv.pooled(x)[0], conv(x, torch.empty(y.numel(), device=DEV), 0.5)

    assert all(torch.equal(a, b) for a, b in zip(passes(layer), passes(fresh)))


def test_packed_weights_of_another_shape_are_refused(pkg):
    layer = pkg.convnet.Conv3x3(_weights(64, 64, 1))
    layer.packed = torch.zeros((9, 64, 32), device=DEV)
    with pytest.raises(ValueError):
        layer(torch.zeros((2, 64, 160, 160), device=DEV))
