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


def _close(a, b):
    return float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


class _Changed(torch.nn.Module):
    """A layer in another's place: its output changed, none of its attributes."""

    def __init__(self, layer, change):
        super().__init__()
        self.layer, self.change = layer, change

    def forward(self, *args, **kwargs):
        return self.change(self.layer(*args, **kwargs))


def test_hooked_and_replaced_generator_layers(pkg):
    """Hooks on a style layer and on the output layers run with what those
    compute, and layers put in their place are called."""
    gen, wp, noises = _generator()
    with torch.no_grad():
        plain = gen.synthesis(wp, noises)
        # the output layers' own images add up to the maps
        seen = []
        handles = [c.register_forward_hook(lambda m, a, out: seen.append(out)) for c in gen.to_rgb]
        gen.synthesis(wp, noises)
        assert len(seen) == len(gen.to_rgb)
        total = seen[0]
        for t in seen[1:]:
            total = pkg.convnet.upsample2(total) + t
        assert _close(total, plain)
        for h in handles:
            h.remove()
        # a hook that changes a style (by more than a factor, which the
        # demodulation takes out), and a layer that does in the affine's place
        affine = gen.convs[2].affine
        handle = affine.register_forward_hook(lambda m, a, out: out.roll(1, 1))
        hooked = gen.synthesis(wp, noises)
        handle.remove()
        gen.convs[2].affine = _Changed(affine, lambda out: out.roll(1, 1))
        replaced = gen.synthesis(wp, noises)
        gen.convs[2].affine = affine
        kept = affine.weight.clone(), affine.bias.clone()
        affine.weight.copy_(kept[0].roll(1, 0))
        affine.bias.copy_(kept[1].roll(1, 0))
        want = gen.synthesis(wp, noises)
        assert _close(hooked, want) and _close(replaced, want) and not _close(want, plain)
        affine.weight.copy_(kept[0])
        affine.bias.copy_(kept[1])
        # whole layers in place of others, called as before
        gen.to_rgb[3], gen.convs[4] = (_Changed(c, lambda out: out) for c in (gen.to_rgb[3], gen.convs[4]))
        assert _close(gen.synthesis(wp, noises), plain)


@pytest.mark.parametrize("layer", [0, 1, 3, 7, 9])
def test_hooked_and_replaced_feature_layers(pkg, layer):
    """The feature vector without a gradient: every layer's hooks run, with the
    layer's whole output, and what they return counts."""
    from svbrdf_amd import materialgan as MG
    net = MG.VGGLoss(torch.device(DEV), [0.1, 0.2, 0.3, 0.4])
    image = torch.rand((2, 3, 96, 80), generator=torch.Generator().manual_seed(layer)).to(DEV)
    with torch.no_grad():
        x, seen, conv = net.normalize(image), [], net.convs[layer]
        handle = conv.register_forward_hook(lambda m, a, out: seen.append(out.shape[1]))
        net.compute_feature_vector(x)
        net.load(image)
        assert seen == [conv.cout] * 2
        handle.remove()
        handle = conv.register_forward_hook(lambda m, a, out: out * 1.5)
        hooked = net.compute_feature_vector(x)
        net.load(image)
        assert torch.equal(net.im_feature, hooked)
        handle.remove()
        net.convs[layer] = _Changed(conv, lambda out: out * 1.5)
        replaced = net.compute_feature_vector(x)
    net.convs[layer] = conv
    net.convs[layer].register_forward_hook(lambda m, a, out: out * 1.5)
    want = net.compute_feature_vector(x.clone().requires_grad_(True)).detach()
    assert _close(hooked, want) and _close(replaced, want)
