"""16-channel convolutions on grids of more than 512 small tiles, where the
kernel with 16 x 8 x 8 tiles takes over, at sizes around its tiles: one voxel
past a tile, one short of it, one row thin, exact; and the last grid of the
other kernel.  Small integers, so that every sum is exact."""
import numpy as np
import pytest

from oracle import unet_ref as U
from pyro_amd import net as N

pytestmark = pytest.mark.gpu


def _ints(rng, shape, lo=-2, hi=3):
    return rng.integers(lo, hi, shape).astype(np.float32)


@pytest.mark.parametrize("ca", [0, 32])
@pytest.mark.parametrize("shape", [(65, 65, 17), (63, 129, 15), (33, 1, 1024), (1, 33, 1009), (8, 1030, 16),
                                   (64, 64, 32)])
def test_conv16_tiles_exact(ca, shape):
    rng = np.random.default_rng(ca + shape[0])
    half = tuple((s + 1) // 2 for s in shape)
    a = _ints(rng, half + (ca,)) if ca else None
    b = _ints(rng, shape + (16,))
    W = _ints(rng, (16, ca + 16, 27), -1, 2)
    bias = _ints(rng, (16,), -3, 4)
    got = N.debug_conv(ca, 16, 16, a, b, W, bias, relu=True)
    assert np.array_equal(got, U.conv_layer(a, b, W, bias, relu_on=True).astype(np.float32))
    if not ca:
        got = N.debug_conv(0, 16, 16, None, b, W, transposed=True)
        assert np.array_equal(got, U.conv_layer_adj(b, W).astype(np.float32))
