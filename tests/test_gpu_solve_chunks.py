"""The dependency-driven solve's chunks of 16 right-hand sides (up to four beside
each other in a launch, further launches beyond 64): widths around every edge,
against the level launches of the same factor, one column at a time, and with
the backward off-diagonal work in one and in several row chunks."""
import dataclasses
import threading

import numpy as np
import pytest

import rslab_amd as R
from rslab_amd import matgen
from test_gpu_parity import rhs
from test_gpu_solve_dep import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("nrhs", [9, 15, 16, 17, 24, 31, 32, 33, 63, 64, 65, 71, 130])
def test_chunked_solve_equals_level_solve_and_single_columns(case, nrhs):
    a, st = CASES[case]()
    st = dataclasses.replace(st, solve_split=0)
    sym = R.LdltSymbolic.analyze_with(a, st)
    f = sym.factor(a)
    f0 = sym.replan(dataclasses.replace(st, solve_dep=False)).factor(a)
    B = rhs(a, nrhs, 5)
    X, X0 = f.solve_many(B), f0.solve_many(B)
    # the same sums in other groupings: rounding on these well-conditioned cases
    assert np.abs(X - X0).max() <= 1e-11 * np.abs(X0).max()
    assert np.array_equal(f.solve_many(B), X)
    for c in (0, 7, 8, nrhs - 1):  # a column does not depend on its chunk
        assert np.array_equal(f.solve(B[:, c]), X[:, c])


@pytest.mark.parametrize("nrhs", [8, 20, 40])
def test_many_off_diagonal_rows(nrhs):
    """A front of 3000 off-diagonal rows: several backward row chunks."""
    m, k = 90, 3000
    rng = np.random.default_rng(2)
    rows = [np.arange(m + k)]
    cols = [np.arange(m + k)]
    vals = [np.where(np.arange(m + k) % 3 == 0, -60.0, 70.0)]
    r, c = np.meshgrid(np.arange(m + k), np.arange(m), indexing="ij")
    low = r > c
    rows.append(r[low]), cols.append(c[low]), vals.append(rng.uniform(-1, 1, int(low.sum())))
    a = R.CscMatrix.from_triplets(m + k, np.concatenate(rows), np.concatenate(cols), np.concatenate(vals))
    st = R.SolverSettings(relax=None, nemin=1, solve_split=0).with_ordering(R.OrderingMethod.Natural)
    sym = R.LdltSymbolic.analyze_with(a, st)
    f = sym.factor(a)
    f0 = sym.replan(dataclasses.replace(st, solve_dep=False)).factor(a)
    B = rhs(a, nrhs, 9)
    X, X0 = f.solve_many(B), f0.solve_many(B)
    assert np.abs(X - X0).max() <= 1e-11 * np.abs(X0).max()


@pytest.mark.parametrize("split", [None, 0, 1])
@pytest.mark.parametrize("nrhs", [1, 20])
def test_one_parent_of_many_children(nrhs, split):
    """3000 leaves under one front of 200 columns: children with and without
    units of their own, and more terms on a row than one round gathers."""
    m, k = 3000, 200
    rng = np.random.default_rng(4)
    n = m + k
    rows = np.concatenate([np.arange(n)] + [m + rng.integers(j * 50, j * 50 + 50, m) for j in range(4)])
    cols = np.r_[np.arange(n), np.tile(np.arange(m), 4)]
    vals = np.r_[np.where(np.arange(n) < m, 4.0, 200.0), rng.uniform(-1, 1, 4 * m)]
    a = R.CscMatrix.from_triplets(n, rows, cols, vals)
    st = dataclasses.replace(R.SolverSettings().with_ordering(R.OrderingMethod.Amd), solve_split=split)
    sym = R.LdltSymbolic.analyze_with(a, st)
    f = sym.factor(a)
    f0 = sym.replan(dataclasses.replace(st, solve_dep=False)).factor(a)
    B = rhs(a, nrhs, 9)
    X, X0 = f.solve_many(B), f0.solve_many(B)
    assert np.abs(X - X0).max() <= 1e-12 * np.abs(X0).max()
    assert np.abs(a.symv(X) - B).max() <= 1e-11


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_bad_right_hand_side_stays_alone(bad, cplx):
    """A column that holds a NaN or an infinity changes no other column, in its
    own chunk or another one, also where its chunk is padded."""
    a = matgen.grid_laplacian((12, 11, 10), shift=-1.3, diag_imag=np.full(1320, 0.1) if cplx else None)
    st = dataclasses.replace(R.SolverSettings().with_ordering(R.OrderingMethod.MetisND), solve_split=0)
    f = R.LdltSymbolic.analyze_with(a, st).factor(a)
    B = rhs(a, 21, 3)
    X = f.solve_many(B)
    for row in (0, 700, 1319):
        for c in (0, 15, 16, 20):
            C = B.copy()
            C[row, c] = bad
            Y = f.solve_many(C)
            keep = np.arange(21) != c
            assert not np.isfinite(Y[:, c]).all() and np.array_equal(Y[:, keep], X[:, keep])


def test_factors_solve_beside_each_other():
    """Two factors with streams of their own, solved from two threads at once,
    several chunks each: every solve waits only on its own counters."""
    jobs = []
    for cplx, m in ((False, 20), (True, 14)):
        a = matgen.grid_laplacian((m, m, m), shift=-1.3, diag_imag=np.full(m ** 3, 0.1) if cplx else None)
        st = dataclasses.replace(R.SolverSettings().with_ordering(R.OrderingMethod.MetisND), solve_split=0)
        f = R.LdltSymbolic.analyze_with(a, st).factor(a)
        B = rhs(a, 70, 3)
        jobs.append((f, B, f.solve_many(B)))
    same = []

    def work(f, B, X):
        for _ in range(10):
            same.append(np.array_equal(f.solve_many(B), X))

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(same) == 20 and all(same)
