"""The U-Net's forward pass on a grid whose input and output go through the
pinned slots (arrays from 8 MiB), against parts of the grid whose arrays are
below that.  A voxel's output depends on voxels at most 24 planes away (1 + 2
for the level-0 and level-1 decoder convolutions, 8 + 4 + 2 for the encoder's,
and the levels' alignment), and every sum's order is the voxel's own, so a part
that starts at a multiple of four gives the same bits 32 planes from its cuts."""
import numpy as np
import pytest

from pyro_amd.net import Net

pytestmark = pytest.mark.gpu


def test_forward_beyond_the_slot_threshold():
    nz, ny, nx = 132, 130, 130
    rng = np.random.default_rng(3)
    x0 = np.stack((rng.normal(size=(nz, ny, nx)), rng.random((nz, ny, nx)) < 0.9), -1).astype(np.float32)
    x0[nz // 2:, ..., 0] *= 0.5  # the two halves, staged one after the other, differ in kind
    net = Net(seed=2)
    net.set_params(rng.normal(0.0, 0.1, net.n).astype(np.float32))
    y = net.forward(x0)
    assert np.array_equal(y, net.forward(x0))
    assert y.std() > 0.0
    for lo, hi, a, b in ((0, 84, 0, 52), (20, 112, 52, 80), (48, 132, 80, 132)):
        part = net.forward(x0[lo:hi])
        assert np.array_equal(part[a - lo:b - lo], y[a:b]), (lo, hi)
