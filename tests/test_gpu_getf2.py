"""Bunch-Kaufman panels of every width class the blocked panel factorization
branches on (one or two rows per lane, whole and partial sub-blocks, matrix-core
tiles with remainders), against the CPU oracle: dense fronts as one supernode,
with plain steps only, with random pivoting, and with a zero diagonal (2x2
pivots at every place of a sub-block, its last column included)."""
import numpy as np
import pytest

import oracle as O
import rslab_amd as R
from rslab_amd import matgen
from test_gpu_parity import assert_same_factor, check_solution, dense_lower_csc, factor_pair, rhs

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 3, 15, 16, 17, 18, 31, 33, 47, 63, 64, 65, 79, 96, 127, 128, 130, 200]


def front(n, kind, cplx):
    M = matgen.rng_uniform(17 + n, -1, 1, n * n).reshape(n, n)
    if cplx:
        M = M + 1j * matgen.rng_uniform(91 + n, -1, 1, n * n).reshape(n, n)
    M = M + M.T
    if kind == "plain":
        M = M + 2 * n * np.eye(n)
    elif kind == "zero_diagonal":
        M[np.arange(n), np.arange(n)] = 0.0
    return dense_lower_csc(M)


@pytest.mark.parametrize("kind", ["plain", "random", "zero_diagonal"])
@pytest.mark.parametrize("panel_nb", [64, 128])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("wide", [False, True])
def test_panel_widths(kind, panel_nb, cplx, wide):
    for n in WIDTHS:
        if n == 1 and kind == "zero_diagonal":
            continue
        a = front(n, kind, cplx)
        st = R.SolverSettings(wide_flops=0.0 if wide else 1e18).with_ordering(R.OrderingMethod.Natural)
        _, fg, fo, s = factor_pair(a, st.with_panel_nb(panel_nb), panel_nb=panel_nb)
        # entries agree to rounding times the pivots' growth (the same bar as
        # the other dense fronts)
        assert_same_factor(fg.factors(), fo)
        check_solution(a, fg, fo, s, rhs(a, 2, 5))


@pytest.mark.parametrize("cplx", [False, True])
def test_perturbed_pivots_inside_a_sub_block(cplx):
    """PerturbToEps lifts a vanishing pivot wherever it sits in a sub-block."""
    n = 40
    M = np.diag(np.linspace(1.0, 2.0, n)).astype(complex if cplx else float)
    for k in (0, 5, 15, 16, 39):
        M[k, k] = 1e-14
    a = dense_lower_csc(M)
    st = R.SolverSettings(scaling="Identity", wide_flops=0.0).with_ordering(R.OrderingMethod.Natural)
    f = R.LdltSolver.factor_with(a, st.with_pivot(R.ZeroPivotAction.PerturbToEps(1e-8)))
    assert f.n_perturbed() == 5
    d = np.abs(f.factors().d_diag)
    assert np.isclose(np.sort(d)[:5], 1e-8, rtol=1e-12).all() and d[5:].min() >= 1e-8


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("n, i, j", [(20, 10, 3), (40, 20, 3), (40, 39, 0), (40, 20, 20), (64, 63, 0), (100, 70, 5),
                                     (128, 127, 64), (130, 129, 2)])
def test_nan_is_no_candidate(n, i, j, wide, cplx):
    """A NaN entry spreads from its pivot on, but never takes part in a search:
    the other entries of its column are still searched, so interchanges, 2x2
    steps, inertia and the places of the NaNs are the oracle's."""
    rng = np.random.default_rng(n + i)
    M = rng.uniform(-1, 1, (n, n)) + (1j * rng.uniform(-1, 1, (n, n)) if cplx else 0.0)
    M = M + M.T
    M[i, j] = M[j, i] = np.nan
    a = dense_lower_csc(M)
    st = R.SolverSettings(wide_flops=0.0 if wide else 1e18).with_ordering(R.OrderingMethod.Natural)
    st = st.with_pivot(R.ZeroPivotAction.PerturbToEps(1e-8))
    sym = R.LdltSymbolic.analyze_with(a, st)
    fg = sym.factor(a, st).factors()
    fo = O.factor(sym.export(), O.scaled(a, O.onepass_scale(a)), pivot=1, abs_floor=1e-8)
    assert np.array_equal(fg.perm, fo.perm) and np.array_equal(fg.two_by_two, fo.two_by_two)
    assert fg.inertia.as_tuple() == fo.inertia and fg.n_perturbed == fo.n_perturbed
    assert np.array_equal(np.isnan(fg.l_values), np.isnan(fo.l_values))
    assert np.array_equal(np.isnan(fg.d_diag), np.isnan(fo.d_diag))
