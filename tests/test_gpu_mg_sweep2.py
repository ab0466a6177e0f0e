"""Levels whose two sweeps run in one launch (k_mg_sweep2, 16 x 8 x 8 tiles),
with the prolongation before them or as the coarsest level's solve: sizes around the tile, rows of every
remainder of four, the smallest row it takes and one below it, and both sides
of the size where single sweeps take over.  Random solid blocks."""
import pytest

import test_gpu_mg_tail as tail
from test_gpu_poisson import _vcycles_match_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,levels", [
    ((16, 64, 32), 2),    # whole tiles
    ((17, 65, 33), 2),    # one cell past them
    ((33, 65, 33), 3),
    ((31, 63, 31), 3),    # one short
    ((18, 57, 40), 2),
    ((35, 16, 200), 2),
    ((96, 96, 96), 4),    # the last size of whole rows
    ((100, 96, 96), 4),   # single sweeps on level 0
    ((23, 45, 15), 1),    # a coarsest level solved by sweeps, odd rows
    ((24, 46, 15), 1),    # and whole rows
    ((48, 72, 15), 1),
])
def test_two_sweeps_bitwise_equal_oracle(dims, levels):
    _vcycles_match_oracle(dims, levels, blocks=5)


@pytest.mark.parametrize("n", [(5, 120, 90), (4, 120, 90), (3, 120, 90)])
def test_short_rows_with_weighted_boundary(n, monkeypatch):
    """The shortest rows it takes (and one below them) in the preconditioner's
    hierarchy, with the reference and the bound of the tail's test."""
    tail.test_tail_with_weighted_boundary(n, monkeypatch)
