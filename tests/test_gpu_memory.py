"""A call that finds no memory on the device reports it and leaves its handle as
it was: the same call fails again, smaller ones give what they gave before."""
import ctypes as C

import numpy as np
import pytest

import rslab_amd as R
from rslab_amd import matgen
from test_gpu_parity import rhs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
def test_a_solve_without_memory_leaves_the_handle_usable(cplx):
    a = matgen.grid_laplacian((10, 10, 10), shift=-1.3, diag_imag=np.full(1000, 0.1) if cplx else None)
    f = R.LdltSolver.factor_with(a)
    B = rhs(a, 3, 5)
    X = f.solve_many(B)
    hip = C.CDLL("libamdhip64.so.7")
    d = C.c_void_p()
    assert hip.hipMalloc(C.byref(d), C.c_size_t(4096)) == 0
    try:
        for _ in range(2):
            # 400 GB of scratch, more than the card has; refused before anything reads d
            with pytest.raises(R.OutOfMemory):
                f.solve_device(d.value, 50_000_000, d.value)
    finally:
        hip.hipFree(d)
    assert np.array_equal(f.solve_many(B), X)
    f.refactor(a)
    assert np.array_equal(f.solve_many(B), X)
