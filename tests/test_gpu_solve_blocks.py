"""The dependency-driven solve's diagonal blocks: 16x16 inverses used plain, with
one correction, or not at all, by the size of their entries; and taken after
the drop tolerance has changed the panels."""
import dataclasses

import numpy as np
import pytest

import rslab_amd as R
from rslab_amd import matgen
from test_gpu_parity import dense_lower_csc, rhs

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def growing(n, entry, cplx, group=16):
    """L D L^T whose unit-lower L has `entry` below the diagonal of every group
    of 16 columns: L's inverse there grows as (1 - entry)^15."""
    rng = np.random.default_rng(3)
    L = np.eye(n, dtype=complex if cplx else float)
    for c in range(0, n, group):
        m = min(group, n - c)
        L[c:c + m, c:c + m] += entry * np.tril(np.ones((m, m)), -1)
    L += np.tril(rng.uniform(-1e-3, 1e-3, (n, n)), -1)
    d = rng.uniform(1.0, 1.05, n) * (np.exp(0.3j * rng.uniform(-1, 1, n)) if cplx else 1.0)
    return L @ np.diag(d) @ L.T


def largest_inverse_entry(f):
    """Over the 16x16 diagonal tiles of the (single) supernode's L, couplings
    left out, as D holds them."""
    L = np.eye(f.n, dtype=f.l_values.dtype)
    for j in range(f.n):
        L[f.l_row_idx[f.l_col_ptr[j]:f.l_col_ptr[j + 1]], j] = f.l_values[f.l_col_ptr[j]:f.l_col_ptr[j + 1]]
    return max(np.abs(np.linalg.inv(L[c:c + 16, c:c + 16])).max() for c in range(0, f.n, 16))


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("entry, lo, hi", [(-0.01, 1.0, 1.25), (-0.3, 1.25, 64.0), (-0.9, 64.0, 1e5)],
                         ids=["plain", "corrected", "substituted"])
@pytest.mark.parametrize("n", [16, 64, 65, 200])
def test_inverses_of_every_size(entry, lo, hi, n, cplx):
    M = growing(n, entry, cplx)
    a = dense_lower_csc(M)
    st = dataclasses.replace(R.SolverSettings().with_ordering(R.OrderingMethod.Natural), solve_split=0)
    sym = R.LdltSymbolic.analyze_with(a, st)
    f = sym.factor(a)
    assert lo <= largest_inverse_entry(f.factors()) <= hi
    f0 = sym.replan(dataclasses.replace(st, solve_dep=False)).factor(a)
    for k in (1, 17):
        B = rhs(a, k, 4)

        def berr(X):
            return (np.abs(M @ X - B) / (np.abs(M) @ np.abs(X) + np.abs(B))).max()

        # the level launches substitute; a few n eps is substitution's own bound
        assert berr(f.solve_many(B)) <= max(3.0 * berr(f0.solve_many(B)), 2 * n * EPS)


def test_dropped_entries_are_gone_from_the_blocks():
    a = matgen.config3(m=16, nrhs=1)[0]
    st = dataclasses.replace(R.SolverSettings().with_ordering(R.OrderingMethod.MetisND), solve_split=0, drop_tol=1e-2)
    sym = R.LdltSymbolic.analyze_with(a, st)
    f = sym.factor(a)
    f0 = sym.replan(dataclasses.replace(st, solve_dep=False)).factor(a)
    B = rhs(a, 5, 6)
    X, X0 = f.solve_many(B), f0.solve_many(B)
    assert np.abs(X - X0).max() <= 1e-11 * np.abs(X0).max()


# Right-hand sides M X make the substituted values small beside the products
# that the inverse sums, so that a plain product's rounding shows: on the CPU
# model of these systems (test_solve_blocks_model.py) it leaves 12 to 1600 times
# substitution's backward error, the corrected one at most 1.8 times.
CANCELLING = dict(entry=[-0.42, -0.9], n=[16, 64, 65])
CANCELLING_BAR = 3.0


def cancelling(M, k=64):
    rng = np.random.default_rng(1)
    return M @ rng.uniform(-1, 1, (len(M), k)).astype(M.dtype)


def backward_error(M, X, B):
    return (np.abs(M @ X - B) / (np.abs(M) @ np.abs(X) + np.abs(B))).max()


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("entry", CANCELLING["entry"], ids=["corrected", "substituted"])
@pytest.mark.parametrize("n", CANCELLING["n"])
def test_no_tile_loses_digits_to_its_inverse(entry, n, cplx):
    M = growing(n, entry, cplx)
    a = dense_lower_csc(M)
    st = dataclasses.replace(R.SolverSettings().with_ordering(R.OrderingMethod.Natural), solve_split=0)
    sym = R.LdltSymbolic.analyze_with(a, st)
    B = cancelling(M)
    X = sym.factor(a).solve_many(B)
    X0 = sym.replan(dataclasses.replace(st, solve_dep=False)).factor(a).solve_many(B)
    assert backward_error(M, X, B) <= CANCELLING_BAR * backward_error(M, X0, B)


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("n", [1, 15, 17, 32, 33, 48, 49, 63, 81, 100, 127])
def test_last_blocks_of_every_tile_count(n, cplx):
    M = growing(n, -0.3, cplx)
    a = dense_lower_csc(M)
    st = dataclasses.replace(R.SolverSettings().with_ordering(R.OrderingMethod.Natural), solve_split=0)
    sym = R.LdltSymbolic.analyze_with(a, st)
    f = sym.factor(a)
    f0 = sym.replan(dataclasses.replace(st, solve_dep=False)).factor(a)
    B = rhs(a, 17, 4)
    X, X0 = f.solve_many(B), f0.solve_many(B)
    # two substitutions of one factor, each within n eps of |L| |L^-1| (< 4^2 here) times the solution
    assert np.abs(X - X0).max() <= 32 * n * EPS * np.abs(X0).max() * np.linalg.cond(M)
