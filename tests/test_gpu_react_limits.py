"""The reaction's shortcuts for cold gas against the oracle where the terms they
leave out are not zero: a step of no length (q = 0 / 0), no oxygen demand and
unbounded coefficients (0 / 0 and 0 inf).  Bit for bit, NaN where the oracle has NaN."""
import numpy as np
import pytest

import oracle
import pyro_amd as pa
from harness import mini_scene, perturbed_state

pytestmark = pytest.mark.gpu

INF = float("inf")


@pytest.mark.parametrize("dt,word,value", [
    (0.002, None, 0.0),
    (0.0, None, 0.0),
    (0.002, "s_o2", 0.0),
    (0.002, "s_o2", INF),
    (0.002, "dhc", INF),
    (0.002, "soot_form", INF),
    (0.002, "soot_ox", INF),
])
def test_react_bitwise_equal_oracle(dt, word, value):
    scene = mini_scene()
    p = scene.params()
    if word:
        p[word] = value
    sol, st = scene.voxelize(), perturbed_state(scene, 11)
    st["s0"][:, :, ::3, 1:3] = 0.0  # neither fuel nor oxygen in a third of the rows
    sims = []
    for make in (oracle.OSim, pa.Sim):
        sim = make(p, sol, None, 4, scene.get("ignition.until"))
        for name in ("s0", "s1", "u", "v", "w", "sol"):
            sim.write_field(name, st[name])
        sims.append(sim)
    o, g = sims
    for sim in sims:
        sim.begin_step(dt, False)
        for stage in ("solid", "curl", "adv_vel1", "adv_vel2", "adv_s1", "adv_s2", "react"):
            sim.run_stage(stage)
    for name in ("s0", "s1"):
        a, b = g.read_field(name), o.read_field(name)
        assert np.array_equal(np.isnan(a), np.isnan(b)), (name, np.argwhere(np.isnan(a) != np.isnan(b))[:4])
        ok = ~np.isnan(b)
        assert np.array_equal(a[ok], b[ok]), name
    g.abort_step()
