"""Buffers made on first use are zeroed before anything is written to them, also
where the null stream, on which a plain memset runs, is far behind: with some
25 ms of memory fills queued there, what a call wrote has to be still there
when they are done."""
import ctypes as C

import numpy as np
import pytest

import pyro_amd as pa
from harness import mini_scene, perturbed_state
from pyro_amd import _native
from pyro_amd.net import Net
from pyro_amd.poisson import Poisson

pytestmark = pytest.mark.gpu


class _Busy:
    """Fills of a 2 GiB block on the null stream, a third of a millisecond each."""

    def __init__(self):
        self.hip = _native.hip()
        self.hip.hipMalloc.argtypes = [C.c_void_p, C.c_size_t]
        self.hip.hipMemset.argtypes = [C.c_void_p, C.c_int, C.c_size_t]
        self.hip.hipFree.argtypes = [C.c_void_p]
        self.p = C.c_void_p()
        assert self.hip.hipMalloc(C.byref(self.p), 2 << 30) == 0

    def go(self):
        for _ in range(75):
            assert self.hip.hipMemset(self.p, 0, 2 << 30) == 0

    def close(self):
        assert self.hip.hipDeviceSynchronize() == 0
        assert self.hip.hipFree(self.p) == 0


@pytest.fixture
def busy():
    b = _Busy()
    yield b
    b.close()


def _pair(seed, shape=(18, 22, 20)):
    rng = np.random.default_rng(seed)
    x0 = np.stack((rng.normal(size=shape), np.ones(shape)), -1).astype(np.float32)
    return x0, rng.normal(size=shape).astype(np.float32)


def test_dataset_add(busy):
    x0, t = _pair(1)
    a, b = Net(seed=1), Net(seed=1)
    a.dataset_add(x0, t)
    busy.go()
    b.dataset_add(x0, t)
    for p, q in zip(a.dataset_get(0, t.shape), b.dataset_get(0, t.shape)):
        assert np.array_equal(p, q)


def test_train_first_call(busy):
    out = []
    for wait in (False, True):
        net = Net(seed=3)
        for k in range(2):
            net.dataset_add(*_pair(k))
        if wait:
            busy.go()
        out.append((net.train(3, lr=1e-3, seed=5), net.params()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_forward_first_call(busy):
    x0, _ = _pair(4)
    a, b = Net(seed=1), Net(seed=1)
    y = a.forward(x0)
    busy.go()
    assert np.array_equal(b.forward(x0), y)
    assert np.array_equal(b.forward(x0), y)


def test_collect(busy):
    scene = mini_scene()
    sim = pa.Sim(scene.params(), scene.voxelize(), None, 4, scene.get("ignition.until"))
    st = perturbed_state(scene, 2)
    for name in ("s0", "s1", "u", "v", "w", "sol"):
        sim.write_field(name, st[name])
    sim.step(0.004)
    sim.sync()
    P = Poisson(sim.read_field(pa.level_field(0, "flags")), scene.grid().dx)
    net = Net(seed=1)
    net.collect(sim, P, 1e-5)
    busy.go()
    net.collect(sim, P, 1e-5)
    shape = sim.dims[::-1]
    for p, q in zip(net.dataset_get(0, shape), net.dataset_get(1, shape)):
        assert np.array_equal(p, q)


def test_render_pack_first_call(busy):
    scene = mini_scene()
    sim = pa.Sim(scene.params(), scene.voxelize(), None, 4, scene.get("ignition.until"))
    sim.step(0.004)
    sim.sync()
    busy.go()
    sim.render_pack_device()
    sim.render_wait()
    assert busy.hip.hipDeviceSynchronize() == 0
    first = sim.read_field("render")
    sim.render_pack_device()
    sim.render_wait()
    assert np.array_equal(first.view(np.uint16), sim.read_field("render").view(np.uint16))
