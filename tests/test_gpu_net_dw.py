"""Weight gradients of the U-Net's convolutions at the row widths where the
kernel's paths change: one to three 32-voxel steps kept in registers, wider
rows, rows with one voxel in the last step, and fewer rows than splits.
Small integers, so that every sum is exact."""
import numpy as np
import pytest

from oracle import unet_ref as U
from pyro_amd import net as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [(32, 16, 16), (0, 32, 32), (0, 64, 64)])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 32), (3, 5, 33), (4, 3, 64), (2, 6, 65), (3, 3, 96), (2, 3, 97),
                                   (1, 7, 130)])
def test_conv_dw_widths_exact(kind, shape):
    ca, cb, co = kind
    rng = np.random.default_rng(co + shape[2])
    half = tuple((s + 1) // 2 for s in shape)
    a = rng.integers(-2, 3, half + (ca,)).astype(np.float32) if ca else None
    b = rng.integers(-2, 3, shape + (cb,)).astype(np.float32)
    g = rng.integers(-2, 3, shape + (co,)).astype(np.float32)
    dW, db = N.debug_conv_dw(ca, cb, co, a, b, g)
    rW, rb = U.conv_layer_dw(a, b, g, co)
    assert np.array_equal(dW, rW.astype(np.float32))
    assert np.array_equal(db, rb.astype(np.float32))
