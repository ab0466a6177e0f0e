"""Coarsest levels too wide for the tail's column segments and too thin for
anything else (k_mg_tail's sweeps on the owned pairs): two, four and eight pairs
a thread, odd x, rows of two and three cells, and the first size beyond the
limit; bit for bit the oracle."""
import numpy as np
import pytest

import oracle
from pyro_amd.poisson import Poisson

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [
    (1031, 2, 2),   # 2064 pairs, odd x
    (512, 2, 4),    # 2048 pairs: exactly two a thread
    (65, 40, 3),    # 3960: four
    (250, 9, 5),    # 5625: eight
    (171, 12, 6),   # 6192: the first beyond the limit
    (3, 700, 2),
    (2, 1030, 2),
])
def test_thin_levels_bitwise_equal_oracle(dims):
    nx, ny, nz = dims
    rng = np.random.default_rng(6)
    flags = (rng.random((nz, ny, nx)) < 0.05).astype(np.uint32)
    b = rng.normal(size=flags.shape).astype(np.float32)
    b[flags == 1] = 0.0
    phi0 = (rng.normal(size=flags.shape) * 0.01).astype(np.float32)
    P = Poisson(flags, 0.05)
    assert P.levels[0] == 1
    P.set(b=b.astype(np.float64), phi=phi0.astype(np.float64))
    P.set_sealed_projection("never")
    assert P.solve("vcycle", tol=0.0, max_iters=2).vcycles == 2
    m = oracle.OMg(dims, 0.05, 4, flags)
    m.set(0, phi0, b)
    m.vcycles(2)
    ref, _, _ = m.get(0)
    got = P.get().astype(np.float32)
    bad = got.view(np.uint32) != ref.view(np.uint32)
    assert not bad.any(), f"{int(bad.sum())} values differ"
