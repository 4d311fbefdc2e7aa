"""LU panels over every height class of the panel factorization (rows per
thread, groups of columns, the panel in memory), as one dense supernode: with
u = 1 the row order and factors are LAPACK getrf's; with a threshold, L U
reconstructs the matrix and no multiplier exceeds 1 / u."""
import numpy as np
import pytest
import scipy.linalg as sla

import rslab_amd as R

pytestmark = pytest.mark.gpu


def dense_csc(M):
    n = M.shape[0]
    return R.GeneralCsc(n, n * np.arange(n + 1), np.tile(np.arange(n), n), M.T.reshape(-1))


def matrix(n, cplx):
    rng = np.random.default_rng(n)
    M = rng.standard_normal((n, n))
    return M + 1j * rng.standard_normal((n, n)) if cplx else M


def device_lu(M, u):
    a = dense_csc(M)
    st = R.SolverSettings().with_ordering(R.OrderingMethod.Natural).with_pivot_u(u)
    sym = R.LuSymbolic.analyze_with(a, st)
    assert sym.info()["nsuper"] == 1
    g = sym.factor(a, st).factors()
    L, U = g.dense_lu()
    return g, L, U, M * g.d_row[:, None] * g.d_col[None, :]


def check_partial_pivoting(g, L, U, lu, order, n):
    assert np.array_equal(g.perm_row, order)
    # rounding of n-term sums of entries below 1 times the growth of partial pivoting
    tol = 1e-10 * max(1.0, n / 600)
    assert np.abs(L - (np.tril(lu, -1) + np.eye(n))).max() <= tol
    assert np.abs(U - np.triu(lu)).max() <= tol * np.abs(U).max()


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 130, 1023, 1025, 2049, 4104])
def test_partial_pivoting_is_lapack(n):
    g, L, U, A = device_lu(matrix(n, False), 1.0)
    lu, piv = sla.lu_factor(A)
    order = np.arange(n)
    for i, p in enumerate(piv):
        order[[i, p]] = order[[p, i]]
    check_partial_pivoting(g, L, U, lu, order, n)


@pytest.mark.parametrize("n", [1, 2, 16, 17, 65, 300])
def test_complex_partial_pivoting_by_modulus(n):
    """(LAPACK compares |re| + |im|.)"""
    g, L, U, A = device_lu(matrix(n, True), 1.0)
    lu, order = A.copy(), np.arange(n)
    for k in range(n):
        p = k + int(np.argmax(np.abs(lu[k:, k]) ** 2))
        lu[[k, p]], order[[k, p]] = lu[[p, k]], order[[p, k]]
        lu[k + 1:, k] /= lu[k, k]
        lu[k + 1:, k + 1:] -= np.outer(lu[k + 1:, k], lu[k, k + 1:])
    check_partial_pivoting(g, L, U, lu, order, n)


@pytest.mark.parametrize("n,cplx", [(40, False), (40, True), (1100, False), (1100, True), (2100, False), (2100, True)])
@pytest.mark.parametrize("u", [0.0, 0.1, 1.0])
def test_threshold_pivoting_reconstructs(n, cplx, u):
    M = matrix(n, cplx) + 2.0 * np.sqrt(n) * np.eye(n)
    M[n // 2, n // 2] = 1e-6 if u > 0.0 else 1.0
    g, L, U, A = device_lu(M, u)
    P = A[g.perm_row]
    assert np.abs(L @ U - P).max() <= 1e-13 * n * (np.abs(L) @ np.abs(U)).max()
    if u > 0.0:
        assert np.abs(L).max() <= 1.0 / u * (1 + 1e-12)
    else:
        assert np.array_equal(g.perm_row, np.arange(n))
