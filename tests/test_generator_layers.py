"""The generator's style layers and output convolution as single kernels
(csrc/generator.hip) against FP64 torch.

A dot product of K terms is within (K + 2) roundings (2^-24 each) of the sum
of its |terms|, the upsampled skip image four more."""
import ctypes

import numpy as np
import pytest
import torch

from tests import convnet_ref as R

DEV = "cuda:0"
EPS = 2.0 ** -24


def test_generator_layers_refuse_on_the_host(pkg):
    """Null pointers, sizes out of range and short or misaligned buffers are
    refused before any launch."""
    from svbrdf_amd import convnet
    lib, f = pkg._lib.load(), ctypes.c_void_p(0x10000)
    t = np.zeros(2, convnet._STYLE_LAYER)
    t["weight"], t["bias"], t["rows"], t["offset"], t["scale"] = 0x10000, 0x20000, [40, 7], [0, 40], 1.0
    p = t.ctypes.data
    assert lib.svbrdf_style_layers_grad_workspace_bytes(p, 2, 512) == 3 * 512 * 4
    assert lib.svbrdf_style_layers(p, 2, None, 14, 512, f, None) == -1
    assert lib.svbrdf_style_layers(p, 33, f, 14, 512, f, None) == -1
    assert lib.svbrdf_style_layers(p, 2, f, 14, 510, f, None) == -2
    assert lib.svbrdf_style_layers(p, 2, ctypes.c_void_p(0x10004), 14, 512, f, None) == -1
    assert lib.svbrdf_style_layers_grad(p, 2, f, 14, 512, f, f, 3 * 512 * 4 - 1, None) == -3
    t["row"] = [0, 14]
    assert lib.svbrdf_style_layers(p, 2, f, 14, 512, f, None) == -2
    assert lib.svbrdf_torgb(f, 512, 4, 4, f, 10, f, 1.0, None, f, None) == -2
    assert lib.svbrdf_torgb(f, 769, 4, 4, f, 9, f, 1.0, None, f, None) == -2
    assert lib.svbrdf_torgb(f, 512, 5, 4, f, 9, f, 1.0, f, f, None) == -2      # a skip image of half an odd size
    assert lib.svbrdf_torgb(None, 512, 4, 4, f, 9, f, 1.0, None, f, None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("dim,rows", [(512, [512, 9, 256]), (4, [1, 33]), (260, [17] * 20), (1028, [64, 16, 15])])
def test_style_layers(pkg, dim, rows):
    from svbrdf_amd import convnet
    g = torch.Generator().manual_seed(dim + len(rows))
    n_latent = 3
    latent = torch.randn((1, n_latent, dim), generator=g).to(DEV).requires_grad_(True)
    weights = [torch.randn((r, dim), generator=g).to(DEV) for r in rows]
    biases = [torch.randn(r, generator=g).to(DEV) for r in rows]
    layers = [((2 * i) % n_latent, 0.1 + 0.01 * i, 0.5) for i in range(len(rows))]
    out = convnet.StyleLayersFunction.apply(latent, weights, biases, layers)
    x = latent.detach().double().requires_grad_(True)
    want = torch.cat([w.double() @ x[0, r] * s + b.double() * bs for w, b, (r, s, bs) in zip(weights, biases, layers)])
    size = torch.cat([w.double().abs() @ x[0, r].detach().abs() * s + b.double().abs() * bs
                      for w, b, (r, s, bs) in zip(weights, biases, layers)])
    assert bool(((out.double() - want).abs() <= (dim + 4) * EPS * size).all())
    probe = torch.randn(out.shape, generator=g).to(DEV)
    (out * probe).sum().backward()
    (want * probe.double()).sum().backward()
    bound = torch.zeros_like(x.detach())
    for w, (r, s, _), p in zip(weights, layers, probe.split(rows)):
        bound[0, r] += p.double().abs() @ w.double().abs() * s
    assert bool(((latent.grad.double() - x.grad).abs() <= (sum(rows) + 6) * EPS * bound + 1e-30).all())


# one and two pixels per lane, remainders of both, few channels, up to 768
@pytest.mark.gpu
@pytest.mark.parametrize("cin,cout,h,w,skip", [(512, 9, 4, 4, False), (512, 9, 8, 8, True), (3, 1, 5, 7, False),
                                               (128, 9, 256, 256, True), (20, 4, 258, 262, True),
                                               (7, 9, 301, 219, False), (768, 9, 16, 18, True)])
def test_torgb(pkg, cin, cout, h, w, skip):
    from svbrdf_amd import convnet
    g = torch.Generator().manual_seed(cin + h)
    x = torch.randn((1, cin, h, w), generator=g).to(DEV).requires_grad_(True)
    st = (1 + 0.3 * torch.randn((1, cin), generator=g)).to(DEV).requires_grad_(True)
    wt = torch.randn((cout, cin, 1, 1), generator=g).to(DEV)
    sk = torch.randn((1, cout, h // 2, w // 2), generator=g).to(DEV).requires_grad_(True) if skip else None
    probe = torch.randn((1, cout, h, w), generator=g).to(DEV)
    y = convnet.ToRGBFunction.apply(x, st, wt, 0.07, sk)
    (y * probe).sum().backward()
    leaves = [t.detach().double().requires_grad_(True) if t is not None else None for t in (x, st, sk)]

    def ref(xx, ss, kk, ww):
        out = torch.einsum("oc,chw->ohw", ww[:, :, 0, 0] * (ss * 0.07), xx[0])[None]
        return out if kk is None else out + R.upsample2_ref(kk)

    want = ref(*leaves, wt.double())
    (want * probe.double()).sum().backward()
    size = ref(*(t.detach().abs() if t is not None else None for t in leaves), wt.double().abs())
    assert bool(((y.double() - want).abs() <= (cin + 10) * EPS * size).all())
    for got, t in zip((x, st, sk), leaves):
        if got is not None:     # library products: norm-wise, as the convolution's gradients
            assert float((got.grad.double() - t.grad).norm() / t.grad.norm()) <= 1e-5


@pytest.mark.gpu
def test_synthesis_paths_agree(pkg):
    """The generator with the fused small layers against the same generator
    computing each layer's own style and output convolution (the path of a
    generator whose layers are being trained): the maps to 1e-5 of their
    largest value, and a mapped batch of two is refused as before."""
    from svbrdf_amd import materialgan as MG
    gen = MG.StyleGAN2Generator(256, 9, seed=1, device=DEV)
    g = torch.Generator().manual_seed(2)
    wp, noises = torch.randn((1, 14, 512), generator=g).to(DEV), gen.make_noises(g)
    with torch.no_grad():
        a = gen.synthesis(wp, noises)
        gen.convs[3].affine.weight.requires_grad_(True)
        assert gen._styles(wp)[0] is None
        b = gen.synthesis(wp, noises)
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())
        with pytest.raises((ValueError, RuntimeError)):
            gen.synthesis(wp.repeat(2, 1, 1), noises)
