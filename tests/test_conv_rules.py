"""Where the convolutions change kernels: shapes on either side of each line."""
import pytest


@pytest.mark.parametrize("shape,taken", [
    ((1, 4096, 4, 4, 4096), 0), ((1, 2048, 8, 8, 2048), 0), ((9, 512, 8, 8, 512), 0), ((1, 1024, 11, 11, 1024), 0),
    ((1, 64, 32, 32, 2048), 0), ((1, 512, 22, 22, 512), 1), ((2, 512, 16, 16, 512), 1), ((9, 64, 256, 256, 64), 1),
    ((9, 256, 64, 64, 256), 1), ((1, 4096, 64, 64, 4096), 1), ((9, 64, 256, 256, 8), 0), ((9, 31, 256, 256, 64), 0),
    ((1, 512, 16, 16, 512), 0), ((0, 64, 256, 256, 64), 0)])
def test_splitting_packed_weights_for_one_call(pkg, shape, taken):
    """Weights that outweigh the image stay packed: splitting them for the call
    would cost more than it saves."""
    lib = pkg._lib.load()
    assert lib.svbrdf_conv3x3_split_packed_preferred(*shape) == taken
    assert lib.svbrdf_conv3x3_split_preferred(*shape) >= taken


@pytest.mark.gpu
@pytest.mark.parametrize("n,cin,cout,h,w", [(9, 3, 64, 40, 24), (1, 16, 16, 100, 96), (2, 64, 72, 30, 28),
                                            (1, 200, 120, 9, 9), (1, 5, 7, 61, 13), (1, 64, 64, 128, 128)])
def test_slices_of_the_weight_gradient_add_up(pkg, n, cin, cout, h, w):
    """Few values in many slices and many in few, whole trips of eight slices
    and remainders.  Each product is rounded with the running sum, 2^-24 of it
    and of either sign, the slices' sums too: norm-wise four times the square
    root of the pixels."""
    import math
    import torch
    g = torch.Generator().manual_seed(cin)
    x, gz = torch.randn((n, cin, h, w), generator=g).cuda(), torch.randn((n, cout, h, w), generator=g).cuda()
    nb = pkg._lib.query("svbrdf_conv3x3_wgrad_workspace_bytes", n, cin, h, w, cout)
    assert nb > 36 * cin * cout and nb % (36 * cin * cout) == 0      # slices
    gw = pkg.convnet.conv3x3_wgrad(x, gz, cout)
    xp, z = torch.nn.functional.pad(x.double(), (1, 1, 1, 1)), gz.double().transpose(0, 1).flatten(1)
    want = torch.stack([z @ xp[:, :, a:a + h, b:b + w].transpose(0, 1).flatten(1).t().contiguous()
                        for a in range(3) for b in range(3)], -1).view(cout, cin, 3, 3)
    assert float((gw.double() - want).norm() / want.norm()) <= 4 * math.sqrt(n * h * w) * 2.0 ** -24
    assert torch.equal(gw, pkg.convnet.conv3x3_wgrad(x, gz, cout))
