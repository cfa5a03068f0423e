"""Device buffers kept for reuse: what a buffer held before, and which object,
thread or stream had it, never shows in a result.  Products and batched KPM
graphs on matrices that take over the buffers of destroyed ones are compared
with the oracle (1e-12 relative, the FP64 tolerance used elsewhere) and with a
dense recursion (12 moments, 1e-10 of the first)."""
import threading

import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu


def make(nb, lo, hi, per_row, seed):
    from vbcsr_amd import VBCSR
    from vbcsr_amd import workloads as W

    M = W.random_vbcsr(nb, bs_lo=lo, bs_hi=hi, per_row=per_row, seed=seed)
    return M, VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals)


@pytest.mark.parametrize("streams", [False, True])
def test_threads_take_over_buffers(streams):
    import torch

    cases = [(150 + 40 * k, 1 + k % 3, 4 + k % 5, 5 + k, k) for k in range(6)]
    want = []
    for c in cases:
        M, _ = make(*c)
        want.append(O.spgemm(O.Mat.of(M), O.Mat.of(M), 0.0))
    bad = []

    def work(t):
        try:
            st = torch.cuda.Stream() if streams else torch.cuda.current_stream()
            with torch.cuda.stream(st):
                for rep in range(8):
                    k = (t + rep) % len(cases)
                    M, H = make(*cases[k])
                    C = H.spmm(H, 0.0)
                    if not np.array_equal(C.col_ind, want[k].col_ind) or relerr(C.get_values(), want[k].vals) > 1e-12:
                        bad.append((t, rep, k))
                    del H, C
        except Exception as e:  # noqa: BLE001
            bad.append((t, repr(e)))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_batched_graph_of_a_later_batch():
    """Batches of equal buffer sizes and different block sizes, one after
    another: each takes over the addresses of the last, none its graph."""
    from vbcsr_amd import VBCSR, kpm

    for lo, n in ((4, 60), (2, 120), (8, 30), (4, 60), (1, 240)):
        g = np.random.default_rng(lo)
        bs = np.full(n, lo, np.int32)
        hs, vs, dense, x0 = [], [], [], []
        for _ in range(3):
            D = g.standard_normal((n * lo, n * lo))
            D = (D + D.T) / (2.4 * np.sqrt(2 * n * lo))  # spectrum inside [-1, 1]
            rp = np.arange(n + 1) * n
            ci = np.tile(np.arange(n), n).astype(np.int32)
            vals = D.reshape(n, lo, n, lo).transpose(0, 2, 1, 3).ravel()
            H = VBCSR.from_block_csr(bs, rp, ci, vals)
            v = H.create_multivector(1)
            x = g.standard_normal((n * lo, 1))
            v.from_numpy(x)
            hs.append(H), vs.append(v), dense.append(D), x0.append(x)
        got = kpm.kpm_moments_batched(hs, vs, 12, precision="fp64")
        for D, x, mu in zip(dense, x0, got):
            t0, t1, ref = x, D @ x, []
            for _ in range(12):
                ref.append(float((x * t0).sum()))
                t0, t1 = t1, 2 * D @ t1 - t0
            assert np.abs(np.asarray(mu).ravel() - ref).max() < 1e-10 * abs(ref[0])
        del hs, vs
