"""GPU row numeric kernel of real SpGEMM (blocks up to 8 x 8, sparse results)
at the sizes where it can go wrong, against the oracle: every block size, rows
with more than 64 A slots, B rows wider than a step of the work-group, C rows
that need several LDS windows, empty rows, and result rows of one slot.

Tolerances: a C value sums at most 250 x 8 products.  FP64: 2000 x 2^-53 =
2e-13 of the largest partial sum, 1e-12 as elsewhere.  FP32: inputs rounded to
2^-24 and a random walk of 2000 roundings, sqrt(2000) x 2^-24 = 3e-6, 1e-5.
BF16: factors rounded to 2^-9, 2e-2 as elsewhere."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu


def hubs(nb, lo, hi, hub_rows, hub_slots, slots, seed):
    """Random blocks of sizes lo..hi; hub_rows rows of hub_slots slots, one row
    of one slot, two empty rows, the others of `slots` slots."""
    from vbcsr_amd import workloads as W

    g = np.random.default_rng(seed)
    bs = g.integers(lo, hi + 1, nb).astype(np.int32)
    n = np.full(nb, slots)
    where = g.permutation(nb)
    n[where[:hub_rows]] = hub_slots
    n[where[hub_rows]] = 1
    n[where[hub_rows + 1:hub_rows + 3]] = 0
    cols = [np.sort(g.choice(nb, k, replace=False)) for k in n]
    rp = np.concatenate([[0], np.cumsum(n)])
    ci = np.concatenate(cols).astype(np.int32)
    nnz = int((bs[np.repeat(np.arange(nb), n)].astype(np.int64) * bs[ci]).sum())
    return W.BlockCSR(bs, rp.astype(rp.dtype), ci, g.standard_normal(nnz))


SIZES = [(1, 1), (2, 2), (3, 3), (4, 4), (5, 5), (6, 6), (7, 7), (8, 8), (1, 8), (1, 4)]


@pytest.mark.parametrize("numeric,tol", [("fp64", 1e-12), ("fp32", 1e-5), ("bf16", 2e-2)])
@pytest.mark.parametrize("lo,hi", SIZES)
def test_rows(lo, hi, numeric, tol):
    from vbcsr_amd import VBCSR

    M = hubs(700, lo, hi, 3, 250, 5, seed=lo * 10 + hi)
    H = VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals)
    C = H.spmm(H, 0.0, numeric=numeric)
    ref = O.spgemm(O.Mat.of(M), O.Mat.of(M), 0.0)
    assert C.local_block_nnz < 0.15 * M.nb**2  # below the dense paths' fill
    assert np.array_equal(C.row_ptr, ref.row_ptr) and np.array_equal(C.col_ind, ref.col_ind)
    assert relerr(C.get_values(), ref.vals) < tol


@pytest.mark.parametrize("nb", [1, 63, 64, 65, 513])
def test_row_counts(nb):
    """Row counts around the chunks the rows are dealt in; narrow B rows (one
    wave per row) and a skip threshold that drops pairs."""
    from vbcsr_amd import VBCSR

    from vbcsr_amd import workloads as W

    g = np.random.default_rng(nb)
    bs = g.integers(1, 9, nb).astype(np.int32)
    n = min(nb, 3)
    ci = np.concatenate([np.sort(g.choice(nb, n, replace=False)) for _ in range(nb)]).astype(np.int32)
    rows = np.repeat(np.arange(nb), n)
    sizes = bs[rows].astype(np.int64) * bs[ci]
    scale = np.repeat(10.0 ** g.uniform(-4, 0, len(ci)), sizes)
    M = W.BlockCSR(bs, np.arange(nb + 1) * n, ci, g.standard_normal(int(sizes.sum())) * scale)
    H = VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals)
    for thr in (0.0, 1e-2):
        C = H.spmm(H, thr)
        ref = O.spgemm(O.Mat.of(M), O.Mat.of(M), thr)
        assert np.array_equal(C.row_ptr, ref.row_ptr) and np.array_equal(C.col_ind, ref.col_ind)
        assert relerr(C.get_values(), ref.vals) < 1e-12


@pytest.mark.parametrize("lo,hi", [(1, 1), (8, 8), (1, 8), (9, 12)])
@pytest.mark.parametrize("nb", [3, 64, 65, 130])
def test_filled_bf16(nb, lo, hi):
    """Results filled enough for the dense BF16 product: block rows around the
    64 slots of a scatter work-group, and blocks beyond its 8 x 8.  With a
    threshold blocks near it may flip under BF16 rounding: the values are
    compared dense."""
    from vbcsr_amd import VBCSR
    from vbcsr_amd import workloads as W

    M = hubs(nb, lo, hi, nb - 3, max(1, nb // 2), 1, seed=nb + hi)
    H = VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals)
    for thr in (0.0, 1e-3):
        C = H.spmm(H, thr, numeric="bf16")
        ref = O.spgemm(O.Mat.of(M), O.Mat.of(M), thr)
        if nb > 3:
            assert ref.col_ind.size > 0.4 * nb * nb
        if thr == 0.0:
            assert np.array_equal(C.row_ptr, ref.row_ptr) and np.array_equal(C.col_ind, ref.col_ind)
        assert relerr(C.to_dense(), W.BlockCSR(M.bs, ref.row_ptr, ref.col_ind, ref.vals).to_dense()) < 2e-2


@pytest.mark.parametrize("numeric,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
@pytest.mark.parametrize("slots", [2, 12, 24, 40])
def test_filled_results(slots, numeric, tol):
    """Results filled by sparse factors (row kernel) and by filled ones (dense
    panels): the share of multiplication paths decides, 0.25 of all triples."""
    from vbcsr_amd import VBCSR

    M = hubs(40, 1, 8, 37, slots, 1, seed=slots)
    H = VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals)
    for thr in (0.0, 1e-3):
        C = H.spmm(H, thr, numeric=numeric)
        ref = O.spgemm(O.Mat.of(M), O.Mat.of(M), thr)
        if thr == 0.0 or numeric == "fp64":
            assert np.array_equal(C.row_ptr, ref.row_ptr) and np.array_equal(C.col_ind, ref.col_ind)
            assert relerr(C.get_values(), ref.vals) < tol
