"""The term-by-term building blocks of the propagation gradient (basis with its
series, Clenshaw cotangents, sampled outer products) against dense numpy, on
uniform 4 x 4 and variable blocks, around the kernels' sizes: one to 70 terms
(64 contraction entries per register set), one and three columns, rows without
blocks and of more than four.

Tolerances: the recurrences are at most 69 FP64 steps on vectors of norm O(1)
(spectral radius below 1), the outer products sums of 210 terms: 1e-11 of the
largest entry; FP32 vectors round every step once (6e-8 each, at most 69
steps, growing at most linearly in a Chebyshev recurrence inside [-1, 1]):
1e-4."""
import ctypes

import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu


def matrix(kind):
    from vbcsr_amd import VBCSR
    from vbcsr_amd.workloads import BlockCSR

    rng = np.random.default_rng(11)
    nb = 23
    bs = np.full(nb, 4, np.int32) if kind == "quads" else rng.choice(np.array([1, 2, 5, 9], np.int32), size=nb)
    lens = [0, 3, 4, 5, 11]
    cols = [np.sort(rng.choice(nb, size=lens[i % 5], replace=False)) for i in range(nb)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    A = BlockCSR(bs.astype(np.int32), rp, np.concatenate(cols).astype(np.int32), np.zeros(0))
    n = int(A.value_offsets()[-1])
    A.vals = rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)
    D = A.to_dense()
    A.vals /= 1.2 * np.linalg.norm(D, 2)
    return A, VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals), D / (1.2 * np.linalg.norm(D, 2))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("K", [1, 3])
@pytest.mark.parametrize("nt", [1, 2, 3, 17, 70])
@pytest.mark.parametrize("kind", ["quads", "variable"])
def test_terms(kind, nt, K, prec):
    import torch

    from vbcsr_amd.autograd import _lib

    A, H, D = matrix(kind)
    L, h = _lib(), ctypes.c_void_p(H._core.handle)
    tol = 1e-11 if prec == 0 else 1e-4
    dt = torch.complex128 if prec == 0 else torch.complex64
    rng = np.random.default_rng(nt)
    center, half = 0.1, 1.2
    Ht = (D - center * np.eye(A.n)) / half
    X, lam = (rng.standard_normal((A.n, K)) + 1j * rng.standard_normal((A.n, K)) for _ in range(2))
    coef = rng.standard_normal(nt) + 1j * rng.standard_normal(nt)
    t = [X, Ht @ X]
    for n in range(2, nt):
        t.append(2 * Ht @ t[-1] - t[-2])
    t = t[:nt]
    b = [None] * (nt + 2)
    b[nt] = b[nt + 1] = np.zeros_like(lam)
    for n in range(nt - 1, -1, -1):
        b[n] = np.conj(coef[n]) * lam + (1 if n == 0 else 2) * Ht.conj().T @ b[n + 1] - b[n + 2]

    def p(x):
        return ctypes.c_void_p(x.data_ptr())

    cp = np.ascontiguousarray(coef).view(np.float64).ctypes.data_as(ctypes.c_void_p)
    Xd, Ld = (torch.as_tensor(v, device="cuda").to(dt) for v in (X, lam))
    stride = A.n * K + 5
    T = torch.zeros((nt, stride), dtype=dt, device="cuda")
    B = torch.zeros_like(T)
    Y = torch.zeros_like(Xd)
    assert L.vbh_cheb_basis_terms(h, K, p(Xd), K, nt, p(T), stride, cp, p(Y), K, center, half, prec, None) == 0
    assert L.vbh_cheb_adjoint_terms(h, K, p(Ld), K, nt, cp, p(B), stride, center, half, prec, None) == 0
    torch.cuda.synchronize()
    assert relerr(T[:, :A.n * K].cpu().numpy().reshape(nt, A.n, K), np.stack(t)) < tol
    assert relerr(Y.cpu().numpy(), sum(c * v for c, v in zip(coef, t))) < tol
    assert relerr(B[:, :A.n * K].cpu().numpy().reshape(nt, A.n, K), np.stack(b[:nt])) < tol
    if nt == 1:
        return
    G = torch.full((A.nnz,), 0.5, dtype=torch.complex128, device="cuda")
    alpha = np.array([2.0, -1.0])
    assert L.vbh_sddmm_terms(h, K, nt, p(B), stride, p(T), stride, 0.25,
                             alpha.ctypes.data_as(ctypes.c_void_p), p(G), prec, None) == 0
    torch.cuda.synchronize()
    w = np.where(np.arange(nt) == 0, 0.25, 1.0)
    full = (2.0 - 1.0j) * sum(wn * bn @ tn.conj().T for wn, bn, tn in zip(w, b, t)) + 0.5
    off, voff = A.offsets(), A.value_offsets()
    ref = np.concatenate([full[off[i]:off[i + 1], off[j]:off[j + 1]].ravel() for i in range(A.nb)
                          for j in A.col_ind[A.row_ptr[i]:A.row_ptr[i + 1]]])
    assert len(ref) == voff[-1]
    assert relerr(G.cpu().numpy(), ref) < tol
