"""The order in which the step's solid tiles are dealt out: a second batch a
block with a short last group, and a grid below one group; against the solid
stage alone as in test_gpu_solid_tiles, bit for bit."""
import pytest

from test_gpu_solid_tiles import test_solid_tiles_equal_solid_stage as solid_tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell", [0.2, 0.019])
def test_solid_order(cell):
    solid_tiles(cell, True)
