"""reload_textures of an upscale (one kernel, svbrdf_reload_textures) against
the three steps it stands for: textures to 8-bit maps, the Lanczos-4 resize of
each and back, bit for bit; they are themselves pinned to the codec oracle in
test_gpu_codec.py."""
import ctypes

import pytest
import torch

DEV = "cuda:0"


def test_reload_refuses_on_the_host(pkg):
    """Null pointers, a size that does not grow or exceeds the maximum, and
    overlapping buffers are refused before any launch."""
    lib, f = pkg._lib.load(), ctypes.c_void_p(0x10000)
    far = ctypes.c_void_p(1 << 40)
    assert lib.svbrdf_reload_textures(None, 8, far, 16, None) == -1
    assert lib.svbrdf_reload_textures(f, 8, None, 16, None) == -1
    for res, dst in ((8, 8), (8, 4), (0, 4), (4096, 7681)):
        assert lib.svbrdf_reload_textures(f, res, far, dst, None) == -2, (res, dst)
    assert lib.svbrdf_reload_textures(f, 8, ctypes.c_void_p(0x10000 + 9 * 64 * 4 - 4), 16, None) == -1


# both tile sizes (16: few tiles or a scale near 1), partial tiles, one texel,
# odd sizes, strong and slight upscales
@pytest.mark.gpu
@pytest.mark.parametrize("src,dst", [(1, 2), (1, 40), (3, 17), (16, 32), (37, 74), (64, 65), (100, 317), (301, 602),
                                     (256, 730), (700, 737), (725, 1009)])
def test_reload_is_the_three_steps(pkg, src, dst):
    from svbrdf_amd import svbrdf_io
    g = torch.Generator().manual_seed(src * 1000 + dst)
    t = torch.rand((1, 9, src, src), generator=g) * 2.4 - 1.2       # past the range: the clips count
    t[0, 3:5] *= 0.6
    t[0, 4, 0, 0] = float("nan")
    t[0, 0, -1, -1] = float("inf")
    t = t.to(DEV)
    got = svbrdf_io.reload_textures(t, dst)
    want = svbrdf_io.textures_from_maps_u8(*svbrdf_io.maps_u8_from_textures(t), dst)
    assert got.shape == want.shape == (1, 9, dst, dst)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    # a strided, batch-less input goes the same way
    wide = torch.zeros((9, src, 2 * src), device=DEV)
    wide[:, :, ::2] = t[0]
    assert torch.equal(svbrdf_io.reload_textures(wide[:, :, ::2], dst).view(torch.int32), want.view(torch.int32))
