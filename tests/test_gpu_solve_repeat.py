"""A solve starts the next V-cycle's first sweeps before it knows whether the
iteration was its last.  What they leave must not reach the next solve: solves
one after the other on one handle, ended by the tolerance, by the iteration
limit and at the first look, against the same solves on fresh handles, bit for
bit.  Sizes: the whole hierarchy in one workgroup, two sweeps a launch, and
single sweeps on level 0."""
import numpy as np
import pytest

from pyro_amd.poisson import Poisson

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(12, 10, 11), (33, 47, 35), (100, 96, 96)])
@pytest.mark.parametrize("method", ["mgpcg", "refine"])
def test_solves_do_not_see_the_last_ones_sweeps(dims, method):
    nx, ny, nz = dims
    rng = np.random.default_rng(4)
    flags = np.zeros((nz, ny, nx), np.uint32)
    flags[2:4, 3:6, 2:7] = 1
    probs = []
    for tol, iters in ((1e-5, 50), (0.0, 2), (1e9, 50), (1e-7, 50), (0.0, 1)):
        b = rng.normal(size=flags.shape)
        b[flags == 1] = 0.0
        probs.append((b, tol, iters))
    one = Poisson(flags, 0.1)
    for b, tol, iters in probs:
        fresh = Poisson(flags, 0.1)
        for P in (one, fresh):
            P.set(b=b, phi=np.zeros_like(b))
        i1, i2 = one.solve(method, tol=tol, max_iters=iters), fresh.solve(method, tol=tol, max_iters=iters)
        assert (i1.iterations, i1.vcycles, i1.rel_resid) == (i2.iterations, i2.vcycles, i2.rel_resid)
        assert np.array_equal(one.get().view(np.uint64), fresh.get().view(np.uint64))
        fresh.close()
