"""Refinement reaches 1e-9 on every grid that test_gpu_solve_pairs lists (there a
solve that does not is skipped)."""
import pytest

from test_gpu_solve_pairs import test_solution_matches_fp64_oracle as solution

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 5, 3), (8, 8, 12), (9, 7, 11), (16, 17, 19), (17, 16, 20), (34, 21, 18)])
def test_refinement_converges(dims):
    try:
        solution(dims, "refine")
    except pytest.skip.Exception as e:
        pytest.fail(str(e))
