"""Coarsest levels with columns too long for the column solve (more than 21
cells) that fit the tail with eight pairs a thread: one segment short, odd x,
nearly all threads and nearly all of the LDS; bit for bit the oracle."""
import pytest

from test_gpu_poisson import _vcycles_match_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,levels", [
    ((48, 9, 22), 1),
    ((40, 9, 28), 1),
    ((23, 10, 50), 1),
    ((12, 15, 80), 1),
    ((56, 9, 32), 1),
    ((88, 19, 44), 2),  # 44x10x22 under a finer level
])
def test_long_columns_bitwise_equal_oracle(dims, levels):
    _vcycles_match_oracle(dims, levels, blocks=5)
