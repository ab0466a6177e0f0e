"""Large host arrays through the pinned slots: sizes below and above the
threshold, one chunk more than the slots, a last chunk of one element, and
two handles used from two threads at once, all byte for byte."""
import threading

import numpy as np
import pytest

from pyro_amd.poisson import Poisson

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(64, 64, 64), (128, 128, 64), (128, 128, 257), (97, 131, 211)])
def test_round_trip_exact(dims):
    nx, ny, nz = dims
    rng = np.random.default_rng(nx)
    P = Poisson(np.zeros((nz, ny, nx), np.uint32), 0.01)
    for _ in range(2):
        b, phi = rng.normal(size=(2, nz, ny, nx))
        P.set(b=b, phi=phi)
        assert np.array_equal(P.get_rhs(), b)
        assert np.array_equal(P.get(), phi)


def test_two_threads():
    rng = np.random.default_rng(5)
    shape = (128, 128, 128)
    bad = []

    def work(seed):
        P = Poisson(np.zeros(shape, np.uint32), 0.01)
        for k in range(4):
            phi = np.random.default_rng(10 * seed + k).normal(size=shape)
            P.set(phi=phi)
            if not np.array_equal(P.get(), phi):
                bad.append((seed, k))
        P.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    P = Poisson(np.zeros(shape, np.uint32), 0.01)  # after the last handle gave the slots back
    phi = rng.normal(size=shape)
    P.set(phi=phi)
    assert np.array_equal(P.get(), phi)
