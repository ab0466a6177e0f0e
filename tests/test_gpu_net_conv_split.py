"""Convolutions whose output channels are split over blocks where a grid has few
tiles: on both sides of each line of that rule (a part of the channels a block,
half of them, all of them), with part tiles in x, y and z.  Small integers, so
that every sum is exact."""
import numpy as np
import pytest

from oracle import unet_ref as U
from pyro_amd import net as N

pytestmark = pytest.mark.gpu


def _ints(rng, shape, lo=-2, hi=3):
    return rng.integers(lo, hi, shape).astype(np.float32)


@pytest.mark.parametrize("kind", [(0, 16, 32), (0, 32, 32), (0, 32, 64), (0, 64, 64), (64, 32, 32)])
@pytest.mark.parametrize("shape", [(7, 11, 18), (30, 77, 20), (33, 81, 33)])  # 12, 320 and 567 tiles
def test_conv_split_exact(kind, shape):
    ca, cb, co = kind
    rng = np.random.default_rng(co + shape[0])
    half = tuple((s + 1) // 2 for s in shape)
    a = _ints(rng, half + (ca,)) if ca else None
    b = _ints(rng, shape + (cb,))
    W = _ints(rng, (co, ca + cb, 27), -1, 2)
    bias = _ints(rng, (co,), -3, 4)
    got = N.debug_conv(ca, cb, co, a, b, W, bias, relu=True)
    assert np.array_equal(got, U.conv_layer(a, b, W, bias, relu_on=True).astype(np.float32))


@pytest.mark.parametrize("kind", [(32, 16, 16), (0, 16, 32), (0, 32, 32), (0, 32, 64), (0, 64, 64), (64, 32, 32)])
@pytest.mark.parametrize("shape", [(7, 11, 18), (30, 77, 20), (33, 81, 33)])
def test_conv_input_gradient_split_exact(kind, shape):
    ca, cb, co = kind
    rng = np.random.default_rng(co + shape[0] + 1)
    W = _ints(rng, (co, ca + cb, 27), -1, 2)
    g = _ints(rng, shape + (co,))
    got = N.debug_conv(ca, cb, co, None, g, W, transposed=True)
    assert np.array_equal(got, U.conv_layer_adj(g, W).astype(np.float32))
