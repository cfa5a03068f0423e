"""Further edges of the matrix-core and vector-ALU kernels: fused steps on
ragged 4 x 4 rows, graphs of batches that take over each other's buffers, the
refusal of precision 2 where no kernel has it, one complex128 column around the
row count that decides its kernel, and FP32 row products with a threshold.

Tolerances as elsewhere: FP64 1e-11 of the first moment or series, 1e-12 of a
product, FP32 storage 2e-5 over 21 moments and 2e-6 of a product (64 products
of values of order one, each rounded three times to 2^-24)."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu


def symmetric(bs, keep, seed):
    """Symmetric matrix of the kept blocks, spectrum inside [-1, 1]."""
    from vbcsr_amd.workloads import BlockCSR

    g = np.random.default_rng(seed)
    nb, n = len(bs), int(bs.sum())
    D = g.standard_normal((n, n))
    D = np.where(np.repeat(np.repeat(keep, bs, 0), bs, 1), D + D.T, 0.0)
    D /= 1.05 * np.abs(np.linalg.eigvalsh(D)).max()
    off = np.concatenate([[0], np.cumsum(bs)])
    rows, cols = np.nonzero(keep)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nb))]).astype(np.int32)
    vals = np.concatenate([D[off[i]:off[i + 1], off[j]:off[j + 1]].ravel() for i, j in zip(rows, cols)])
    return BlockCSR(bs.astype(np.int32), rp, cols.astype(np.int32), vals)


def vb(A):
    from vbcsr_amd import VBCSR

    return VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals)


@pytest.mark.parametrize("nb", [3, 6, 37])
def test_quad_steps_ragged(nb):
    """Fused steps with dots where the four rows of a wave differ in length,
    one of them empty."""
    from vbcsr_amd import kpm

    g = np.random.default_rng(nb)
    keep = np.triu(g.random((nb, nb)) < min(1.0, 7.0 / nb), 0)
    keep[0, :] = True  # one long row and column
    keep = keep | keep.T
    keep[1, :] = keep[:, 1] = False
    A = symmetric(np.full(nb, 4), keep, nb)
    assert len(set(np.diff(A.row_ptr))) > 1
    H, m = vb(A), O.Mat.of(A)
    for K in (1, 2, 5, 10, 19):
        V = H.create_multivector(K)
        V.set_random(5, normalize=False)
        v0 = np.array(V.to_numpy())
        for mode, code in (("one", 1), ("two", 2)):
            ref = O.kpm_moments(m, v0, 21, mode=code)
            for prec, tol in (("fp64", 1e-11), ("fp32", 2e-5), ("mixed", 2e-5)):
                assert relerr(kpm.kpm_moments(H, V, 21, mode=mode, precision=prec), ref) < tol, (K, mode, prec)


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("mixed", 2e-5), ("fp32", 2e-5)])
@pytest.mark.parametrize("K", [2, 8, 17])
def test_batched_graphs_of_later_batches(K, prec, tol):
    """Batches of equal vector sizes on 4 x 4 blocks, small uniform blocks and
    variable blocks in turn: each takes over the addresses of the last, none
    its graph."""
    from vbcsr_amd import kpm

    n = 120
    variable = np.resize(np.array([1, 3, 5, 7, 8], np.int32), 25)
    kinds = [np.full(30, 4), np.full(60, 2), variable, np.full(30, 4), np.full(120, 1), np.full(40, 3), variable]
    for q, bs in enumerate(kinds):
        assert bs.sum() == n
        As = [symmetric(bs, np.ones((len(bs), len(bs)), bool), 10 * q + h) for h in range(3)]
        hs, vs = [vb(A) for A in As], []
        for h, H in enumerate(hs):
            v = H.create_multivector(K)
            v.set_random(q + h, normalize=False)
            vs.append(v)
        for _ in range(2):
            got = kpm.kpm_moments_batched(hs, vs, 12, precision=prec)
            for A, v, mu in zip(As, vs, got):
                ref = O.kpm_moments(O.Mat.of(A), np.asarray(v.to_numpy()), 12, mode=2)
                assert relerr(mu, ref) < tol, (q, K)
        del hs, vs


@pytest.mark.parametrize("sizes", [[2], [4], [1, 4, 9]])
def test_precision_2_refused(sizes):
    """Adjoints and more than 64 columns have no mixed kernel: refused, and
    the result is not touched."""
    import torch

    bs = np.resize(np.array(sizes), 12)
    H = vb(symmetric(bs, np.ones((12, 12), bool), 1))
    for K, adjoint in ((3, True), (65, False), (65, True)):
        x = torch.ones((int(bs.sum()), K), dtype=torch.float64, device="cuda")
        y = torch.full_like(x, 7.0)
        with pytest.raises(Exception):
            H._core.spmm_raw(K, x.data_ptr(), K, y.data_ptr(), K, 2, adjoint)
        torch.cuda.synchronize()
        assert (y == 7.0).all()


@pytest.mark.parametrize("nb", [1, 1023, 1024, 1027])
def test_one_complex_column(nb):
    import torch
    from vbcsr_amd.workloads import BlockCSR

    g = np.random.default_rng(nb)
    lens = np.array([0, 1, 4, 5, 17, 10])[np.arange(nb) % 6] if nb > 1 else np.array([1])
    ci = np.concatenate([np.sort(g.choice(nb, k, replace=False)) for k in lens]).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    A = BlockCSR(np.full(nb, 4, np.int32), rp, ci, g.uniform(-1, 1, 16 * len(ci)) + 1j * g.uniform(-1, 1, 16 * len(ci)))
    H, m = vb(A), O.Mat.of(A)
    x = g.standard_normal((A.n, 1)) + 1j * g.standard_normal((A.n, 1))
    for prec, dt, tol in ((0, torch.complex128, 1e-12), (1, torch.complex64, 2e-6)):
        for adjoint in (False, True):
            xd = torch.as_tensor(x, device="cuda").to(dt)
            y = torch.full_like(xd, 7.0)
            H._core.spmm_raw(1, xd.data_ptr(), 1, y.data_ptr(), 1, prec, adjoint)
            torch.cuda.synchronize()
            ref = O.spmm_adjoint(m, x) if adjoint else O.spmm(m, x)
            assert relerr(y.cpu().numpy(), ref) < tol, (prec, adjoint)
    coef = g.standard_normal(8) + 1j * g.standard_normal(8)
    xv = H.create_multivector(1)
    xv.from_numpy(x)
    y = np.asarray(memoryview(H._core.cheb_apply(xv._core, coef, 0.1, 30.0, 0)))
    assert relerr(y, O.cheb_apply(m, x, coef, 0.1, 30.0)) < 1e-11


def test_row_products_fp32_threshold():
    """FP32 row products with a skip and filter threshold, compared dense
    (blocks near the threshold may flip: their values are below it)."""
    from vbcsr_amd import workloads as W

    thr = 1e-3
    M = W.random_vbcsr(300, bs_lo=1, bs_hi=8, per_row=6, seed=3)
    H = vb(M)
    C = H.spmm(H, thr, numeric="fp32")
    assert H.spmm_stats[2] < 0.5 * M.nb**2  # not the dense panels
    ref = O.spgemm(O.Mat.of(M), O.Mat.of(M), thr)
    R = W.BlockCSR(M.bs, ref.row_ptr, ref.col_ind, ref.vals).to_dense()
    assert np.abs(C.to_dense() - R).max() < max(1e-5 * np.abs(R).max(), 1.1 * thr)
