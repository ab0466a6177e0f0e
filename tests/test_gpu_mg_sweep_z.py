"""Sweeps of levels beyond 12 million cells (k_mg_sweep_z: 32 x 8 tiles walked
along z in chunks of 30 planes), at sizes that leave part tiles in x and y and
a last chunk of one plane, or of twelve, and on a grid of long rows.  Random
solid blocks."""
import pytest

from test_gpu_poisson import _vcycles_match_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,levels", [
    ((228, 230, 241), 4),
    ((256, 256, 192), 4),
    ((3000, 66, 62), 4),
])
def test_sweep_along_z_bitwise_equal_oracle(dims, levels):
    _vcycles_match_oracle(dims, levels)
