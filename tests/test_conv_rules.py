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
