"""The complex field's two cmod forms (product blocks and their sums; the
gathered tiles for levels above the product-buffer cap) against the oracle: a
damped grid of ragged sizes and a dense 2-level front whose updaters leave
remainders in every tile."""
import numpy as np
import pytest

import rslab_amd as R
from rslab_amd import matgen
from test_gpu_parity import assert_same_factor, check_solution, factor_pair, rhs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [None, 0, "half"])
@pytest.mark.parametrize("method", [R.FactorMethod.LeftLooking, R.FactorMethod.RightLooking])
@pytest.mark.parametrize("dims", [(5, 4, 3), (13, 11, 9), (16, 16, 16)])
def test_cmod_forms_match_the_oracle(cap, method, dims):
    n = int(np.prod(dims))
    delta = matgen.rng_uniform(3, -0.01, 0.01, n)
    eta = 0.1 + matgen.rng_uniform(4, 0.0, 0.4, n)
    a = matgen.grid_laplacian(dims, shift=-1.2, diag_real=delta, diag_imag=eta)
    st = R.SolverSettings().with_ordering(R.OrderingMethod.MetisND).with_method(method)
    if cap == "half":
        cap = R.LdltSymbolic.analyze_with(a, st).cmod_elems_max() // 2
    _, fg, fo, s = factor_pair(a, st.with_cmod_cap(cap))
    assert_same_factor(fg.factors(), fo)
    check_solution(a, fg, fo, s, rhs(a, 3, 11))
