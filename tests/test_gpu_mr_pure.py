"""Level-2 blocks among level-2 blocks, whose rows read the sums of their couplings: with
every block of level 2 (domain faces, ragged or not, in all directions), with a lone refined box
inside, and with one at a corner, so that waves hold such blocks alone, mixed with others,
and none.  The exact solutions and bars are those of the row layout's tests.
"""
import pytest

import test_gpu_mr_rows as rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,boxes", [
    ((32, 28, 24), ()), ((37, 30, 41), ()), ((52, 36, 44), ([24, 8, 20, 32, 16, 28],)),
    ((44, 41, 36), ([0, 0, 0, 12, 12, 8],))])
def test_pure_level_2_blocks_match_the_exact_solution(dims, boxes):
    rows.test_fast_solves_match_the_exact_solution(dims, 2, boxes)
