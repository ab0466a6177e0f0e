"""The step's solid tiles, dealt out to at most 1024 blocks in batches of eight,
against the solid stage alone, which has one block a tile: fewer tiles than
blocks, one batch a block, and a second batch.  Solid cells are scattered over
the whole grid, some about to burn out, so that every block and batch has some;
two steps, so that burnt cells are cleared.  Bit for bit, statistics included."""
import numpy as np
import pytest

import pyro_amd as pa
from harness import VEC4, VEL, perturbed_state, pool_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell", [0.1, 0.04, 0.03])
@pytest.mark.parametrize("stats", [False, True])
def test_solid_tiles_equal_solid_stage(cell, stats):
    scene = pool_scene(cell)
    sims = []
    st = perturbed_state(scene, 5)
    rng = np.random.default_rng(1)
    sol = st["sol"]
    here = np.argwhere(sol[..., 1] > 0.0)
    cells = rng.random(sol.shape[:3]) < 0.004
    sol[cells] = sol[tuple(here[0])]
    sol[cells, 3] = rng.uniform(300.0, 700.0, int(cells.sum()))
    burn = cells & (rng.random(cells.shape) < 0.3)
    # fuel just above the burn-out mass (Params' 42nd word)
    sol[burn, 1] = np.float32(1.0001) * np.frombuffer(scene.params().bytes(), np.float32)[41]
    for _ in range(2):
        sim = pa.Sim(scene.params(), scene.voxelize(), None, 4, scene.get("ignition.until"))
        for name in ("s0", "s1", "u", "v", "w"):
            sim.write_field(name, st[name])
        sim.write_field("sol", sol)
        sim.write_field(pa.level_field(0, "phi"), st["phi"])
        sims.append(sim)
    a, b = sims
    for _ in range(2):
        a.step(0.002, stats)
        b.begin_step(0.002, stats)
        for stg in pa.STAGES:
            if stg != "resid" or stats:
                b.run_stage(stg)
        b.end_step()
        for n in VEC4 + VEL + ("flags",):
            assert np.array_equal(a.read_field(n), b.read_field(n)), n
        if stats:
            assert np.array_equal(a.read_stats().raw, b.read_stats().raw)
