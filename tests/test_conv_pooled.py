"""A convolution that writes its output's 2x2 averages itself: the same bits as
the layer and the pooling one after the other, at odd sizes, ragged channels
and with a scaled copy; and the shapes and modes that run one after the other."""
import pytest
import torch

DEV = "cuda:0"


def test_which_shapes_pool(pkg):
    q = lambda *a: bool(pkg._lib.query("svbrdf_conv3x3_split_pools", *a))   # noqa: E731
    assert q(9, 64, 256, 256, 64) and q(9, 128, 128, 128, 128)
    assert not q(9, 64, 1, 200000, 64) and not q(1, 64, 16, 16, 64) and not q(9, 3, 256, 256, 64)
    assert not q(1, 512, 32, 32, 512)                    # K split over blocks


@pytest.mark.gpu
@pytest.mark.parametrize("n,cin,cout,h,w", [(9, 64, 64, 96, 97), (9, 64, 64, 131, 70), (5, 128, 100, 90, 101),
                                            (9, 128, 128, 128, 128)])
@pytest.mark.parametrize("act", ["none", "relu", "lrelu"])
def test_against_the_layer_and_the_pooling(pkg, n, cin, cout, h, w, act):
    C, g = pkg.convnet, torch.Generator().manual_seed(4)
    assert pkg._lib.query("svbrdf_conv3x3_split_pools", n, cin, h, w, cout)
    layer = C.Conv3x3(torch.randn((cout, cin, 3, 3), generator=g).to(DEV) / (9 * cin) ** 0.5,
                      torch.randn(cout, generator=g).to(DEV), act=act)
    x = torch.randn((n, cin, h, w), generator=g).to(DEV)
    y = layer(x)
    ref = C.avgpool2(y)
    tap = torch.empty(y.numel(), device=DEV)
    pool, out = layer.pooled(x, True, tap, 0.7)
    assert torch.equal(pool, ref) and torch.equal(out, y) and torch.equal(tap.view_as(y), y * 0.7)
    pool, out = layer.pooled(x, False)
    assert torch.equal(pool, ref) and out is None
    # with a gradient: the layer, then the pooling
    xg = x.requires_grad_(True)
    pool, out = layer.pooled(xg, False)
    assert pool.requires_grad and torch.equal(pool.detach(), ref) and torch.equal(out.detach(), y)


@pytest.mark.gpu
def test_not_finite_values_pool_as_before(pkg):
    g = torch.Generator().manual_seed(6)
    layer = pkg.convnet.Conv3x3(torch.randn((64, 64, 3, 3), generator=g).to(DEV))
    x = torch.randn((9, 64, 96, 96), generator=g).to(DEV)
    x[0, 0, 7, 8], x[3, 5, 95, 95] = float("inf"), float("nan")
    pool, _ = layer.pooled(x, False)
    ref = pkg.convnet.avgpool2(layer(x))
    assert bool(((pool == ref) | (pool.isnan() & ref.isnan())).all())
