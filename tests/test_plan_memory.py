"""How a factor splits the device memory beside its panels (rsl_symbolic_scratch,
the numbers the factor itself allocates by): the cmod's product buffer and
operand pool only where they leave the solves their room, none of either where
they do not fit."""
import numpy as np
import pytest

import rslab_amd as R
from rslab_amd import matgen


def planned(dims=(14, 13, 12), **kw):
    a = matgen.grid_laplacian(dims, shift=-1.2)
    return R.LdltSymbolic.analyze_with(a, R.SolverSettings(**kw).with_ordering(R.OrderingMethod.MetisND))


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("precision", [R.Precision.FP64, R.Precision.FP32_SCHUR])
@pytest.mark.parametrize("cap", [None, 0, 1000])
def test_buffers_fit_whatever_is_free(cplx, precision, cap):
    sym = planned(precision=precision, cmod_cap=cap)
    most = sym.scratch(1 << 45, cplx)
    assert most["cmod_elems"] == (sym.cmod_elems_max() if cap is None else cap)
    # the reduced-precision products read no operand pool
    assert (most["operand_bytes"] > 0) == (most["cmod_elems"] > 0 and (cplx or precision == R.Precision.FP64))
    last = 0
    for free in [0] + [int(2 ** e) for e in np.arange(8, 36, 0.25)]:
        s = sym.scratch(free, cplx)
        assert s["pack_bytes"] == most["pack_bytes"]
        taken = s["cmod_bytes"] + s["operand_bytes"]
        if s["cmod_elems"] == 0:
            assert taken == 0
        else:
            assert s["operand_bytes"] == most["operand_bytes"]
            assert s["cmod_bytes"] <= free // 4
            assert taken + s["pack_bytes"] <= free - free // 4
        assert s["cmod_elems"] >= last
        last = s["cmod_elems"]
    assert last == most["cmod_elems"]


def test_a_complex_factor_without_room_for_the_pool_takes_the_gathered_form():
    """Room for the buffer (under a quarter of the free memory) but not for the
    pool: the products are left to the gathered cmod, which needs neither."""
    sym = planned()
    need = sym.scratch(1 << 45, True)
    s = sym.scratch(need["operand_bytes"] + need["pack_bytes"], True)
    assert s["cmod_elems"] == s["cmod_bytes"] == s["operand_bytes"] == 0


def test_scratch_arguments_are_checked():
    sym = planned()
    with pytest.raises(R.InvalidInput):
        sym.scratch(-1)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("relax", [(256, 64), None])
def test_the_solve_pack_follows_the_widths(cplx, relax):
    """A supernode's diagonal blocks take the 16x16 tiles that its columns
    reach: 2 for up to 16 columns, 14 for 64, whatever the tree (a band in its
    natural order runs every supernode, narrow ones too, in the
    dependency-driven part)."""
    n = 3000
    a = R.CscMatrix.from_triplets(n, np.r_[np.arange(n), np.arange(3, n)], np.r_[np.arange(n), np.arange(n - 3)],
                                  np.r_[np.full(n, 4.0), np.ones(n - 3)])
    st = R.SolverSettings(relax=relax, nemin=4, solve_split=0).with_ordering(R.OrderingMethod.Natural)
    sym = R.LdltSymbolic.analyze_with(a, st)
    tiles = 0
    for w in sym.export().sn_ncol:
        for c in range(0, w, 64):
            nt = -(-min(w - c, 64) // 16)
            tiles += 2 * nt + nt * (nt - 1) // 2
    assert sym.scratch(1 << 40, cplx)["pack_bytes"] == tiles * 256 * (16 if cplx else 8)
