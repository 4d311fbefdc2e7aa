"""LU solve steps (64 rows, up to 16 right-hand sides a pass) and the panels'
off-diagonal parts at their edges: fronts of m own columns over k more rows and
columns, against a dense solve, each right-hand side independent of the others."""
import numpy as np
import pytest

import rslab_amd as R

pytestmark = pytest.mark.gpu


def arrow(m, k, cplx):
    """m dense leading rows and columns over a tail that couples only to them."""
    n = m + k
    rng = np.random.default_rng(n)
    r, c = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    keep = (r < m) | (c < m) | (r == c)
    v = rng.uniform(-1, 1, (n, n)) + (1j * rng.uniform(-1, 1, (n, n)) if cplx else 0.0)
    M = np.where(keep, v, 0.0) + np.diag(np.where(np.arange(n) < m, 0.0, 4.0 * m))
    cols, rows = np.nonzero(keep.T)  # column by column
    ptr = np.concatenate([[0], np.cumsum(keep.sum(0))])
    return M, R.GeneralCsc(n, ptr, rows, M[rows, cols])


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("u", [0.1, 1.0])
@pytest.mark.parametrize("m, k", [(1, 1), (15, 3), (16, 63), (63, 64), (64, 65), (65, 1), (130, 200)])
def test_fronts_and_widths(m, k, u, cplx):
    M, a = arrow(m, k, cplx)
    st = R.SolverSettings().with_ordering(R.OrderingMethod.Natural).with_pivot_u(u)
    f = R.LuSymbolic.analyze_with(a, st).factor(a, st)
    rng = np.random.default_rng(1)
    cond = np.linalg.cond(M)
    for nrhs in (1, 4, 5, 8, 9, 16, 17, 33):
        B = rng.uniform(-1, 1, (m + k, nrhs)) + (1j * rng.uniform(-1, 1, (m + k, nrhs)) if cplx else 0.0)
        X = f.solve_many(B)
        # a stable elimination's bound with the growth that 1 / u allows in practice
        err = np.abs(X - np.linalg.solve(M, B)).max() / np.abs(X).max()
        assert err <= 100 * (m + k) * cond * np.finfo(float).eps / u
        for c in {0, nrhs // 2, nrhs - 1}:
            assert np.array_equal(f.solve_many(B[:, c:c + 1])[:, 0], X[:, c])


@pytest.mark.parametrize("cplx", [False, True])
def test_a_bad_right_hand_side_stays_alone(cplx):
    M, a = arrow(70, 30, cplx)
    st = R.SolverSettings().with_ordering(R.OrderingMethod.Natural)
    f = R.LuSymbolic.analyze_with(a, st).factor(a, st)
    B = np.random.default_rng(2).uniform(-1, 1, (100, 9)) + (0j if cplx else 0.0)
    X = f.solve_many(B)
    B[3, 4] = np.nan
    Y = f.solve_many(B)
    keep = np.arange(9) != 4
    assert np.isnan(Y[:, 4]).any() and np.array_equal(Y[:, keep], X[:, keep])
