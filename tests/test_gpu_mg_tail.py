"""The multigrid tail (the levels that run in one workgroup, k_mg_tail) at
the sizes where its mappings change: one to eight pairs per thread, odd
sizes, one to three levels, level 0 included with its warm start."""
import numpy as np
import pytest

import mg_numpy
from pyro_amd.poisson import Poisson
from test_gpu_poisson import _vcycles_match_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,levels", [
    ((9, 9, 5), 1),      # 225 pairs, one per thread, odd x
    ((12, 24, 12), 1),   # two per thread
    ((15, 30, 14), 1),   # four, a short last z segment, odd x
    ((40, 50, 8), 1),    # eight (2000 columns: not the column solve's)
    ((16, 30, 16), 2),   # both levels in the tail
    ((17, 28, 16), 2),   # the same with odd sizes
    ((33, 47, 35), 3),   # two of three levels, odd sizes
    ((31, 30, 24), 2),   # the coarsest alone
])
def test_tail_bitwise_equal_oracle(dims, levels):
    _vcycles_match_oracle(dims, levels, blocks=5)


@pytest.mark.parametrize("n", [(33, 47, 35), (24, 20, 26)])
def test_tail_with_weighted_boundary(n, monkeypatch):
    """The preconditioner hierarchy (neighbours outside the box weigh
    2 2^l / (2^l + 1) on level l), one refinement step from zero, against the
    float64 restatement of the V-cycle.  An FP32 V-cycle rounds each of the
    160 solve passes and eight sweeps by 2^-24 of the values they move, and
    the passes contract: 200 * 2^-24 = 1.2e-5 relative bounds the sum."""
    nx, ny, nz = n
    rng = np.random.default_rng(3)
    flags = np.zeros((nz, ny, nx), np.uint32)
    flags[4:7, 3:9, 5:11] = 1
    b = rng.normal(size=flags.shape)
    b[flags == 1] = 0.0
    h = 0.05
    P = Poisson(flags, h)
    P.set_sealed_projection("never")
    P.set(b=b.astype(np.float32).astype(np.float64), phi=np.zeros_like(b))
    P.solve("refine", tol=0.0, max_iters=1)
    shapes = [flags.shape]
    for _ in range(P.levels[1] - 1):
        shapes.append(tuple((d + 1) // 2 for d in shapes[-1]))
    plain = mg_numpy.nb_sum

    def weighted(p, f):
        s, c = plain(p, f)
        inside = np.zeros_like(p)
        fl = f == 0
        for ax in range(3):
            up = [slice(None)] * 3
            dn = [slice(None)] * 3
            up[ax], dn[ax] = slice(1, None), slice(None, -1)
            inside[tuple(dn)] += fl[tuple(up)]
            inside[tuple(up)] += fl[tuple(dn)]
        l = shapes.index(p.shape)
        w = 1.0 if l == 0 else float(np.float32(2.0 * 2.0 ** l / (2.0 ** l + 1.0)))
        return s, inside + w * (c - inside)

    monkeypatch.setattr(mg_numpy, "nb_sum", weighted)
    # float32 spacings as the levels hold them
    ref = mg_numpy.vcycle(np.zeros_like(b), b.astype(np.float32).astype(np.float64), flags,
                          float(np.float32(h)), P.levels[1])
    got = P.get()
    fluid = flags == 0
    err = np.linalg.norm((got - ref)[fluid]) / np.linalg.norm(ref[fluid])
    assert err < 1.2e-5, err
