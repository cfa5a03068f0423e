"""What products share: the LDS limit of the row kernel between threads, and the
device memory left beside large factors.  Against the oracle or dense numpy at
1e-12 of the largest entry, the FP64 tolerance used elsewhere."""
import ctypes
import threading

import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu


def test_window_sizes_of_two_threads():
    """Products whose LDS windows differ (a few KB, and more than the 64 KB a
    kernel may use without asking), at the same time on two streams."""
    import torch
    from vbcsr_amd import VBCSR
    from vbcsr_amd import workloads as W

    ms = [W.random_vbcsr(60, bs_lo=1, bs_hi=3, per_row=3, seed=1), W.random_vbcsr(2500, bs_lo=7, bs_hi=8, per_row=60, seed=2)]
    want = [O.spgemm(O.Mat.of(m), O.Mat.of(m), 0.0) for m in ms]
    bad = []

    def work(t, reps):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                H = VBCSR.from_block_csr(ms[t].bs, ms[t].row_ptr, ms[t].col_ind, ms[t].vals)
                for rep in range(reps):
                    C = H.spmm(H, 0.0)
                    if rep % 10 == 0 and relerr(C.get_values(), want[t].vals) > 1e-12:
                        bad.append((t, rep))
        except Exception as e:  # noqa: BLE001
            bad.append((t, repr(e)))

    ts = [threading.Thread(target=work, args=a) for a in ((0, 120), (1, 20))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("numeric,tol", [("fp64", 1e-12), ("fp32", 1e-5), ("bf16", 2e-2)])
@pytest.mark.parametrize("nbc", [300, 9000])
def test_few_paths(nbc, numeric, tol):
    """Fewer multiplication paths than B has blocks: no column records; with
    and without a column map, rows of C in one window and in several, skips."""
    from vbcsr_amd import VBCSR
    from vbcsr_amd import workloads as W

    g = np.random.default_rng(nbc)
    bs = g.integers(1, 9, nbc).astype(np.int32)

    def pattern(lens):
        cols = [np.sort(g.choice(nbc, k, replace=False)) for k in lens]
        rows = np.repeat(np.arange(nbc), lens)
        ci = np.concatenate(cols).astype(np.int32)
        sizes = bs[rows].astype(np.int64) * bs[ci]
        scale = np.repeat(10.0 ** g.uniform(-4, 0, len(ci)), sizes)
        rp = np.concatenate([[0], np.cumsum(lens)])
        return W.BlockCSR(bs, rp, ci, g.standard_normal(int(sizes.sum())) * scale)

    few = np.zeros(nbc, np.int64)
    few[[0, 3, nbc // 2, nbc - 1]] = [1, 5, 70, 2]
    A, B = pattern(few), pattern(np.full(nbc, 30))
    HA, HB = (VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals) for M in (A, B))
    for thr in (0.0, 1e-2):
        C = HA.spmm(HB, thr, numeric=numeric)
        ref = O.spgemm(O.Mat.of(A), O.Mat.of(B), thr)
        if thr == 0.0 or numeric == "fp64":
            assert np.array_equal(C.row_ptr, ref.row_ptr) and np.array_equal(C.col_ind, ref.col_ind)
            assert relerr(C.get_values(), ref.vals) < tol


def test_beside_large_factors():
    """A product that fits the memory left beside its factors runs, although
    the column records of its right factor (128 MB here) would not fit: 90 MB
    are left, the product itself needs about a tenth of that."""
    import torch
    from vbcsr_amd import VBCSR
    from vbcsr_amd import workloads as W
    from vbcsr_amd.autograd import _lib

    g = np.random.default_rng(0)
    nb, slots = 1024, 1000
    bs = np.full(nb, 8, np.int32)
    ci = np.concatenate([np.sort(g.choice(nb, slots, replace=False)) for _ in range(nb)]).astype(np.int32)
    B = W.BlockCSR(bs, np.arange(nb + 1) * slots, ci, g.random(nb * slots * 64) - 0.5)
    rp = np.concatenate([[0], np.full(nb, nb)])  # one full row
    A = W.BlockCSR(bs, rp, np.arange(nb, dtype=np.int32), g.random(nb * 64) - 0.5)
    HA, HB = (VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals) for M in (A, B))
    ref = HA.spmm(HB, 0.0).get_values()  # with all the memory there is; the kernels are loaded
    L = _lib()
    huge = ctypes.c_void_p()
    L.vbh_malloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    assert L.vbh_malloc(ctypes.byref(huge), 1 << 45) != 0  # fails, and gives back the buffers kept for reuse
    torch.cuda.empty_cache()
    hold = []
    try:
        for _ in range(4):  # what other buffers give back appears a little later
            free = torch.cuda.mem_get_info()[0]
            if free > 92 << 20:
                hold.append(torch.empty(free - (90 << 20), dtype=torch.uint8, device="cuda"))
                torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] < 120 << 20
        C = HA.spmm(HB, 0.0)
        assert C.local_block_nnz == nb
        got = C.get_values()
    finally:
        hold.clear()
        torch.cuda.empty_cache()
    assert np.array_equal(got, ref)
    row = A.vals.reshape(nb, 8, 8).transpose(1, 0, 2).reshape(8, nb * 8)
    cols = np.zeros((nb * 8, 16))  # the first two block columns of B
    for k in range(nb):
        for q in range(2):
            at = np.searchsorted(ci[k * slots:(k + 1) * slots], q)
            if at < slots and ci[k * slots + at] == q:
                p = (k * slots + at) * 64
                cols[8 * k:8 * k + 8, 8 * q:8 * q + 8] = B.vals[p:p + 64].reshape(8, 8)
    want = (row @ cols).reshape(8, 2, 8).transpose(1, 0, 2).ravel()
    assert relerr(got[:128], want) < 1e-12
