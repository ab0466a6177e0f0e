"""Coarse flags and neighbour codes of all levels (two launches a hierarchy, a
third and a fourth beyond four and seven levels), with solids thick enough to
be solid on every coarse level, on odd grids whose last coarse cells lie partly
outside."""
import numpy as np
import pytest

import mg_numpy
import oracle
from pyro_amd.poisson import Poisson

pytestmark = pytest.mark.gpu


def _flags(dims):
    nx, ny, nz = dims
    f = np.zeros((nz, ny, nx), np.uint32)
    f[:, : ny // 3, nx // 2:] = 1          # a block to the sides of the box
    f[nz - 9:, ny // 2:, : nx // 3] = 1
    f[3, 1, 1] = 1
    return f


@pytest.mark.parametrize("dims", [(64, 48, 32), (67, 45, 51), (130, 101, 99), (33, 32, 31)])
def test_thick_solids_bitwise_equal_oracle(dims):
    f = _flags(dims)
    rng = np.random.default_rng(2)
    b = np.where(f == 1, 0.0, rng.normal(size=f.shape)).astype(np.float32)
    P = Poisson(f, 0.05)
    P.set_sealed_projection("never")
    P.set(b=b.astype(np.float64), phi=np.zeros(f.shape))
    P.solve("vcycle", tol=0.0, max_iters=2)
    m = oracle.OMg(dims, 0.05, 4, f)
    m.set(0, np.zeros(f.shape, np.float32), b)
    m.vcycles(2)
    got = P.get().astype(np.float32)
    assert np.array_equal(got.view(np.uint32), m.get(0)[0].view(np.uint32))


@pytest.mark.parametrize("dims", [(100, 70, 90), (131, 140, 129)])
def test_deep_hierarchy_flags(dims, monkeypatch):
    """The preconditioner's hierarchy (five and six levels), one step from zero
    against the float64 V-cycle, which derives the flags level by level; bound
    as in test_tail_with_weighted_boundary (a wrong flag moves phi by percents)."""
    f = _flags(dims)
    rng = np.random.default_rng(3)
    b = np.where(f == 1, 0.0, rng.normal(size=f.shape)).astype(np.float32).astype(np.float64)
    P = Poisson(f, 0.05)
    P.set_sealed_projection("never")
    P.set(b=b, phi=np.zeros_like(b))
    P.solve("refine", tol=0.0, max_iters=1)
    assert P.levels[1] >= 5
    shapes = [f.shape]
    for _ in range(P.levels[1] - 1):
        shapes.append(tuple((d + 1) // 2 for d in shapes[-1]))
    plain = mg_numpy.nb_sum

    def weighted(p, fl):
        s, c = plain(p, fl)
        inside = np.zeros_like(p)
        for ax in range(3):
            up, dn = [slice(None)] * 3, [slice(None)] * 3
            up[ax], dn[ax] = slice(1, None), slice(None, -1)
            inside[tuple(dn)] += (fl == 0)[tuple(up)]
            inside[tuple(up)] += (fl == 0)[tuple(dn)]
        l = shapes.index(p.shape)
        w = 1.0 if l == 0 else float(np.float32(2.0 * 2.0 ** l / (2.0 ** l + 1.0)))
        return s, inside + w * (c - inside)

    monkeypatch.setattr(mg_numpy, "nb_sum", weighted)
    ref = mg_numpy.vcycle(np.zeros_like(b), b, f, float(np.float32(0.05)), P.levels[1])
    fluid = f == 0
    err = np.linalg.norm((P.get() - ref)[fluid]) / np.linalg.norm(ref[fluid])
    assert err < 1.2e-5, err
