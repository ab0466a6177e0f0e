"""Gradients through the ReLUs, which the adjoint convolutions apply: a grid
of more than 512 tiles, where the 16-channel layers take the kernel of their
own, with rows, columns and planes that end inside a tile.  Three taps of +-1
per channel and whole numbers for input and upstream gradient make every sum
of a voxel exact in FP32, so that no ReLU and no rounding to bfloat16 goes the
other way than the oracle's; only the sums over the grid round.  These add at
most 2^18 terms in parts of at most 2^10, so their error is below 2^11 * 2^-24
= 1.2e-4 of the terms' size; 1e-3 of the norm leaves room for cancellation."""
import numpy as np
import pytest

from oracle import unet_ref as U
from pyro_amd import net as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(33, 66, 67)])
def test_backward_through_relu_large_grid(shape):
    rng = np.random.default_rng(6)
    p = U.split(np.zeros(U.N_PARAMS))
    for name, co, ci in U.LAYERS:
        for c in range(co):
            p["W" + name][c].flat[rng.choice(27 * ci, 3, replace=False)] = 1, 1, -1
    p["wh"][:] = rng.choice([-1, 1], 16)
    flat = U.join(p).astype(np.float32)
    net = N.Net(seed=5)
    net.set_params(flat)
    m = (rng.random(shape) > 0.15).astype(np.float32)
    x0 = np.stack([rng.integers(-2, 3, shape).astype(np.float32) * m, m], axis=-1)
    gy = rng.integers(-1, 2, shape).astype(np.float32)
    G, GR = N.split_params(net.backward(x0, gy)), U.split(U.backward(flat, x0, gy))
    for k in GR:
        assert np.linalg.norm(G[k] - GR[k]) <= 1e-3 * np.linalg.norm(GR[k]), k
