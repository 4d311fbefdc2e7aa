"""A model of the solve's 16x16 inverses on the CPU: on the systems and
right-hand sides of the device test, an uncorrected inverse product is past that
test's bar and the corrected one is not, so the test fails where the
correction or the substitution is missing."""
import numpy as np
import pytest

from test_gpu_solve_blocks import CANCELLING, CANCELLING_BAR, backward_error, cancelling, growing


def ldl(M):
    """L and D of M = L D L^T without interchanges."""
    n = len(M)
    L, d, A = np.eye(n, dtype=M.dtype), np.zeros(n, dtype=M.dtype), M.copy()
    for k in range(n):
        d[k] = A[k, k]
        L[k + 1:, k] = A[k + 1:, k] / d[k]
        A[k + 1:, k + 1:] -= np.outer(L[k + 1:, k], A[k + 1:, k])
    return L, d


def lower_solve(L, B, how):
    X = B.copy()
    for c in range(0, len(L), 16):
        T, b = L[c:c + 16, c:c + 16], X[c:c + 16].copy()
        m = len(T)
        if how == "substituted":
            for i in range(m):
                b[i] -= T[i, :i] @ b[:i]
        else:
            inv = np.eye(m, dtype=L.dtype)
            for i in range(m):
                inv[i] -= T[i, :i] @ inv[:i]
            x = inv @ b
            b = x + inv @ (b - T @ x) if how == "corrected" else x
        X[c:c + 16] = b
        X[c + 16:] -= L[c + 16:, c:c + 16] @ b
    return X


def solve(M, B, how):
    L, d = ldl(M)
    y = lower_solve(L, B, how) / d[:, None]
    back = np.ascontiguousarray(L[::-1, ::-1].T)  # L^T, last row first
    return lower_solve(back, y[::-1], how)[::-1]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("entry", CANCELLING["entry"])
@pytest.mark.parametrize("n", CANCELLING["n"])
def test_the_bar_tells_the_plain_product_from_the_corrected_one(entry, n, cplx):
    M = growing(n, entry, cplx)
    B = cancelling(M)
    e = {how: backward_error(M, solve(M, B, how), B) for how in ("plain", "corrected", "substituted")}
    assert e["plain"] > CANCELLING_BAR * e["substituted"]
    assert e["corrected"] <= CANCELLING_BAR * e["substituted"]
