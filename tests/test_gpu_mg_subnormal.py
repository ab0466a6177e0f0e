"""The pressure solve where quotients come out subnormal: the division by a
count takes its slow path there, which every kernel must reach.  phi and b are
scaled so that h^2 b is subnormal; column solves of 20 and 21 cells in both
layouts, the tail, two sweeps a launch.  Bit-identical to the oracle."""
import numpy as np
import pytest

import oracle
from pyro_amd.poisson import Poisson

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(15, 52, 20), (14, 43, 20), (12, 60, 21), (15, 52, 21), (18, 28, 11), (30, 104, 40),
                                  (9, 9, 5), (33, 47, 35), (23, 45, 15)])
@pytest.mark.parametrize("scale", [1e-36, 3e-39])
def test_subnormal_quotients_bitwise_equal_oracle(dims, scale):
    nx, ny, nz = dims
    rng = np.random.default_rng(7)
    flags = np.zeros((nz, ny, nx), np.uint32)
    flags[1:3, 2:5, 3:7] = 1
    b = (rng.normal(size=flags.shape) * scale).astype(np.float32)
    b[flags == 1] = 0.0
    phi0 = (rng.normal(size=flags.shape) * 0.0025 * scale).astype(np.float32)
    h = 0.05
    P = Poisson(flags, h)
    P.set(b=b.astype(np.float64), phi=phi0.astype(np.float64))
    P.set_sealed_projection("never")
    P.solve("vcycle", tol=0.0, max_iters=2)
    m = oracle.OMg((nx, ny, nz), h, 4, flags)
    m.set(0, phi0, b)
    m.vcycles(2)
    ref, _, _ = m.get(0)
    got = P.get().astype(np.float32)
    assert np.any((np.abs(ref) > 0) & (np.abs(ref) < 1.1754944e-38))
    bad = got.view(np.uint32) != ref.view(np.uint32)
    assert not bad.any(), f"{int(bad.sum())} values differ"
