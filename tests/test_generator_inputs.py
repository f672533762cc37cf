"""What the generator's and the feature network's callers may hand over besides
freshly allocated tensors and untouched layers."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _generator():
    from svbrdf_amd import materialgan as MG
    gen = MG.StyleGAN2Generator(256, 9, seed=1, device=DEV)
    g = torch.Generator().manual_seed(2)
    return gen, torch.randn((1, 14, 512), generator=g).to(DEV), gen.make_noises(g)


@pytest.mark.parametrize("offset", [1, 2, 3, 4])
def test_latent_and_weights_at_any_address(pkg, offset):
    """A W+ that is a view into a larger buffer, and style layers whose weights
    are views of one: the same maps as from aligned copies, to the roundings of
    the layers' other path (1e-5 of the largest value, as between the paths)."""
    gen, wp, noises = _generator()
    room = torch.zeros(wp.numel() + 4, device=DEV)
    view = room[offset:offset + wp.numel()].view(wp.shape)
    view.copy_(wp)
    probe = torch.randn((1, 9, 256, 256), generator=torch.Generator().manual_seed(3)).to(DEV)

    def maps_and_gradient(latent):
        latent = latent.detach().requires_grad_(True)
        out = gen.synthesis(latent, noises)
        (out * probe).sum().backward()
        return out.detach(), latent.grad

    want = maps_and_gradient(wp)
    assert view.data_ptr() % 16 == 4 * (offset % 4) and view.is_contiguous()
    got = maps_and_gradient(view)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    affine = gen.convs[3].affine
    flat = torch.zeros(affine.weight.numel() + 4, device=DEV)
    weight = flat[offset:offset + affine.weight.numel()].view(affine.weight.shape)
    weight.copy_(affine.weight)
    affine.weight = torch.nn.Parameter(weight, requires_grad=False)
    with torch.no_grad():
        out = gen.synthesis(wp, noises)
    assert float((out - want[0]).abs().max()) <= 1e-5 * float(want[0].abs().max())
