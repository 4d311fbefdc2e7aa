"""The wide path's deep-row replay in the complex field (16 panel columns a pass
on the matrix cores, 64 rows a unit) against the CPU oracle: panels that end
inside a pass, units that end inside 64 rows, and 2x2 pivots across passes."""
import numpy as np
import pytest

import rslab_amd as R
from rslab_amd import matgen
from test_gpu_parity import assert_same_factor, check_solution, factor_pair, rhs

pytestmark = pytest.mark.gpu


def arrow(m, k, zero_diagonal):
    """m dense leading columns over k rows that couple to nothing else: one
    supernode of m columns and k off-diagonal rows, and the rest."""
    n = m + k
    r, c = np.meshgrid(np.arange(n), np.arange(m), indexing="ij")
    low = r > c
    rows = np.concatenate([np.arange(n), r[low]])
    cols = np.concatenate([np.arange(n), c[low]])
    v = matgen.rng_uniform(17 + n, -1, 1, rows.size) + 1j * matgen.rng_uniform(910 + n, -1, 1, rows.size)
    if zero_diagonal:
        v[:m] = 0.0
    v[m:n] += 4 * m
    return R.CscMatrix.from_triplets(n, rows, cols, v)


@pytest.mark.parametrize("zero_diagonal", [False, True])
@pytest.mark.parametrize("panel_nb", [64, 128])
@pytest.mark.parametrize("m, k", [(17, 1), (63, 64), (64, 65), (65, 63), (97, 130), (144, 7), (200, 300)])
def test_replay_matches_the_oracle(m, k, panel_nb, zero_diagonal):
    a = arrow(m, k, zero_diagonal)
    st = R.SolverSettings(relax=None, nemin=1, wide_flops=0.0).with_ordering(R.OrderingMethod.Natural)
    _, fg, fo, s = factor_pair(a, st.with_panel_nb(panel_nb), panel_nb=panel_nb)
    assert_same_factor(fg.factors(), fo)
    check_solution(a, fg, fo, s, rhs(a, 2, 5))
