"""Rows of a real product that need several LDS windows, one work-group a window,
some, or all of them in turn (32,768 work-groups over the block rows), with and
without a column map, against the oracle; 1e-12 in FP64, 1e-5 in FP32 as in the
other row-kernel tests."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr
from test_gpu_spgemm_rows import hubs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("numeric,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
@pytest.mark.parametrize("nb,lo,hi", [(600, 8, 8), (4000, 1, 8), (8000, 5, 8), (9000, 1, 8), (17000, 7, 8), (33000, 8, 8)])
def test_windows(nb, lo, hi, numeric, tol):
    from vbcsr_amd import VBCSR

    M = hubs(nb, lo, hi, 2, 400, 4, seed=nb)
    H = VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals)
    for thr in (0.0, 0.5) if numeric == "fp64" else (0.0,):
        C = H.spmm(H, thr, numeric=numeric)
        ref = O.spgemm(O.Mat.of(M), O.Mat.of(M), thr)
        longest = np.diff(ref.row_ptr).max() * lo
        assert longest > 1.1 * 80 * 1024 / (8 if numeric == "fp64" else 4) / (hi | 1) or lo == 1
        assert np.array_equal(C.row_ptr, ref.row_ptr) and np.array_equal(C.col_ind, ref.col_ind)
        assert relerr(C.get_values(), ref.vals) < tol
