"""What products share: the LDS limit of the row kernel between threads.  Against
the oracle at 1e-12 of the largest entry, the FP64 tolerance used elsewhere."""
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
