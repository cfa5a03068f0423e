"""SpMM, KPM steps and Chebyshev series of uniform 4 x 4 blocks at the edges of
their kernel: block-row counts around the four rows of a wave, rows without
blocks and of unequal, long lengths, and column counts around the slices and
lane groups, in every storage precision, against the oracle.

Tolerances: every sum runs in FP64 over at most 160 products of values of order
one, so FP64 results agree to 1e-12 of the largest entry; FP32 storage rounds
each matrix value and X entry once (6e-8 each) and the result once, so 2e-6."""
import ctypes

import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu


def ragged(nb, seed, cplx, lens):
    """nb block rows of 4 x 4 blocks with the given row lengths (capped at nb)."""
    from vbcsr_amd.workloads import BlockCSR

    rng = np.random.default_rng(seed)
    cols = [np.sort(rng.choice(nb, size=min(lens[i % len(lens)], nb), replace=False)) for i in range(nb)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    ci = np.concatenate(cols).astype(np.int32) if rp[-1] else np.zeros(0, np.int32)
    v = rng.uniform(-1, 1, 16 * len(ci))
    if cplx:
        v = v + 1j * rng.uniform(-1, 1, len(v))
    return BlockCSR(np.full(nb, 4, np.int32), rp, ci, v)


def vb(A):
    from vbcsr_amd import VBCSR

    return VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5, 17, 63])
def test_spmm_edges(nb, cplx):
    import torch

    A = ragged(nb, 100 + nb, cplx, [0, 1, 3, 4, 5, 16, 17, 33, 40])
    H, m = vb(A), O.Mat.of(A)
    rng = np.random.default_rng(nb)
    for K in (2, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17, 31, 33, 64):
        X = rng.standard_normal((A.n, K))
        if cplx:
            X = X + 1j * rng.standard_normal(X.shape)
        ref = O.spmm(m, X)
        for prec in (0, 1, 2):
            low = prec == 1
            dt = (np.complex64 if low else np.complex128) if cplx else (np.float32 if low else np.float64)
            for ld in (K, K + 1):
                x = torch.zeros((A.n, ld), dtype=getattr(torch, np.dtype(dt).name), device="cuda")
                x[:, :K] = torch.as_tensor(X.astype(dt), device="cuda")
                y = torch.full_like(x, 7.0)
                H._core.spmm_raw(K, x.data_ptr(), ld, y.data_ptr(), ld, prec, False)
                torch.cuda.synchronize()
                got = y.cpu().numpy()
                assert relerr(got[:, :K], ref) < (1e-12 if prec == 0 else 2e-6), (nb, K, prec, ld)
                assert (got[:, K:] == 7.0).all()


@pytest.mark.parametrize("nb", [3, 6, 37])
def test_kpm_steps_ragged(nb):
    from vbcsr_amd import kpm

    A = ragged(nb, 7 * nb, False, [1, 2, 5, 9, 18])
    D = A.to_dense()
    D = (D + D.T) / 2
    D /= 1.05 * np.abs(np.linalg.eigvalsh(D)).max()
    full = ragged(nb, 0, False, [nb])  # every block stored: the symmetric dense matrix
    full.vals = np.concatenate([D[4 * i:4 * i + 4, 4 * j:4 * j + 4].ravel() for i in range(nb) for j in range(nb)])
    H, m = vb(full), O.Mat.of(full)
    for K in (2, 5, 10, 19):
        V = H.create_multivector(K)
        V.set_random(5, normalize=False)
        v0 = np.array(V.to_numpy())
        for mode, code in (("one", 1), ("two", 2)):
            ref = O.kpm_moments(m, v0, 21, mode=code)
            for prec, tol in (("fp64", 1e-11), ("fp32", 2e-5), ("mixed", 2e-5)):
                assert relerr(kpm.kpm_moments(H, V, 21, mode=mode, precision=prec), ref) < tol, (nb, K, mode, prec)


@pytest.mark.parametrize("cplx", [False, True])
def test_chebyshev_series(cplx):
    """The series accumulated in the step's launch (no reference kernel): K = 1
    to 9 columns against the oracle's Chebyshev apply."""
    A = ragged(29, 3, cplx, [2, 7, 0, 19])
    H, m = vb(A), O.Mat.of(A)
    rng = np.random.default_rng(8)
    coef = rng.standard_normal(7) + (1j * rng.standard_normal(7) if cplx else 0j)
    for K in (2, 3, 9):
        X = rng.standard_normal((A.n, K)) + (1j * rng.standard_normal((A.n, K)) if cplx else 0.0)
        xv = H.create_multivector(K)
        xv.from_numpy(X)
        y = np.asarray(memoryview(H._core.cheb_apply(xv._core, coef, 0.1, 30.0, 0)))
        assert relerr(y, O.cheb_apply(m, X, coef, 0.1, 30.0)) < 1e-11, K


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("nb", [1, 3, 4, 6, 17, 50])
def test_one_column(nb, cplx):
    """K = 1, forward and adjoint, contiguous and strided vectors."""
    import torch

    A = ragged(nb, 300 + nb, cplx, [0, 1, 4, 5, 15, 16, 17, 34, 50])
    H, m = vb(A), O.Mat.of(A)
    rng = np.random.default_rng(nb)
    x = rng.standard_normal((A.n, 1)) + (1j * rng.standard_normal((A.n, 1)) if cplx else 0.0)
    for adjoint in (False, True):
        ref = O.spmm_adjoint(m, x) if adjoint else O.spmm(m, x)
        for prec in (0, 1):
            dt = (np.complex64 if prec else np.complex128) if cplx else (np.float32 if prec else np.float64)
            for ld in (1, 3):
                xd = torch.full((A.n, ld), 5.0, dtype=getattr(torch, np.dtype(dt).name), device="cuda")
                xd[:, :1] = torch.as_tensor(x.astype(dt), device="cuda")
                y = torch.full_like(xd, 7.0)
                H._core.spmm_raw(1, xd.data_ptr(), ld, y.data_ptr(), ld, prec, adjoint)
                torch.cuda.synchronize()
                got = y.cpu().numpy()
                assert relerr(got[:, :1], ref) < (1e-12 if prec == 0 else 2e-6), (nb, adjoint, prec, ld)
                assert (got[:, 1:] == 7.0).all()


@pytest.mark.parametrize("cplx", [False, True])
def test_one_column_series_and_moments(cplx):
    from vbcsr_amd import kpm

    A = ragged(31, 4, cplx, [2, 7, 0, 19])
    H, m = vb(A), O.Mat.of(A)
    rng = np.random.default_rng(9)
    coef = rng.standard_normal(8) + (1j * rng.standard_normal(8) if cplx else 0j)
    X = rng.standard_normal((A.n, 1)) + (1j * rng.standard_normal((A.n, 1)) if cplx else 0.0)
    xv = H.create_multivector(1)
    xv.from_numpy(X)
    y = np.asarray(memoryview(H._core.cheb_apply(xv._core, coef, 0.1, 30.0, 0)))
    assert relerr(y, O.cheb_apply(m, X, coef, 0.1, 30.0)) < 1e-11
    ref = O.kpm_moments(m, X, 15, mode=1, center=0.1, half_width=30.0)
    for prec, tol in (("fp64", 1e-11), ("fp32", 2e-5)):
        got = kpm.kpm_moments(H, xv, 15, mode="one", precision=prec, center=0.1, half_width=30.0)
        assert relerr(got, ref) < tol, prec
