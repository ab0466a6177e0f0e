"""One Poisson handle over steps whose solid flags change: the codes, the fluid
count and the sealed pockets have to be those of the flags at hand, as on a
handle made from them."""
import numpy as np
import pytest

import pyro_amd as pa
from harness import mini_scene, perturbed_state
from pyro_amd.poisson import Poisson, step_solve

pytestmark = pytest.mark.gpu


def _sim(scene, st, sol):
    sim = pa.Sim(scene.params(), scene.voxelize(), None, 4, scene.get("ignition.until"))
    for name in ("s0", "s1", "u", "v", "w"):
        sim.write_field(name, st[name])
    sim.write_field("sol", sol)
    sim.write_field(pa.level_field(0, "phi"), st["phi"])
    return sim


def _walls(sol):
    """Solids in other places: a hollow box (a sealed pocket) and a block of wood."""
    out = sol.copy()
    wood = sol[tuple(np.argwhere(sol[..., 1] > 0.0)[0])]
    out[8:16, 24:34, 6:14] = wood
    out[10:14, 26:32, 8:12] = np.float32(0.0)
    out[20:24, 10:13, 18:26] = wood
    return out


def test_solved_steps_follow_the_flags():
    scene = mini_scene()
    st = perturbed_state(scene, 7)
    sols = [st["sol"], st["sol"], _walls(st["sol"]), _walls(st["sol"]), st["sol"]]
    first = _sim(scene, st, sols[0])
    one = Poisson(first.read_field(pa.level_field(0, "flags")), scene.grid().dx)
    for sol in sols:
        out = []
        for handle in (one, None):
            sim = _sim(scene, st, sol)
            P = handle or Poisson(sim.read_field(pa.level_field(0, "flags")), scene.grid().dx)
            info = step_solve(sim, P, 0.004, "mgpcg", tol=1e-6, max_iters=60)
            out.append((info.iterations, info.rel_resid, P.sealed_info(),
                        sim.read_field(pa.level_field(0, "phi")), sim.read_field("u")))
        assert out[0][:3] == out[1][:3]
        assert (out[0][2][0] > 0) == (sol is not st["sol"])  # the pocket, in the changed solids only
        for a, b in zip(out[0][3:], out[1][3:]):
            assert np.array_equal(a, b), np.abs(a - b).max()
