"""Infinities in X reach the rows whose stored blocks meet them, and no others:
a product sums the stored elements only, so what a kernel pads (slots past a
row's last, chunks past a block's width, lists that end inside an instruction)
must not turn an infinity into NaN.  Every column of X holds one infinity in a
row of its own; forward and adjoint, every kernel of the dispatch, around the
column counts of their slices, in every storage precision, against dense numpy
(finite entries to the tolerances used elsewhere: 1e-12 in FP64, 2e-6 with
FP32 storage, of the largest finite entry)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = {
    "one": ([1], 40, [0, 1, 3, 17]),
    "two": ([2], 41, [0, 1, 3, 4, 5, 17]),
    "three": ([3], 40, [0, 1, 3, 17, 5]),
    "three_long": ([3], 40, [17, 40]),
    "many_two": ([2], 8200, [3, 1]),
    "quads": ([4], 39, [0, 1, 3, 4, 5, 16, 17, 33]),
    "edges": ([3, 4, 5, 7, 8, 9], 61, [0, 2, 7, 30]),
    "sixteens": ([15, 16, 17], 33, [1, 5, 33]),
    "mixed": ([1, 4, 9, 13], 60, [0, 4, 50, 60]),
    "up_to_8": ([1, 2, 5, 8], 60, [1, 40, 60]),
    "up_to_8_short": ([1, 2, 5, 8], 60, [0, 1, 3, 9]),
    "long_lists": ([2, 33, 21], 40, [40, 3]),
}


def build(kind, cplx):
    from vbcsr_amd.workloads import BlockCSR

    sizes, nb, lens = KINDS[kind]
    rng = np.random.default_rng(len(kind))
    bs = rng.permutation(np.resize(np.array(sizes, np.int32), nb))
    cols = [np.sort(rng.choice(nb, size=min(lens[i % len(lens)], nb), replace=False)) for i in range(nb)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    A = BlockCSR(bs, rp, np.concatenate(cols).astype(np.int32), np.zeros(0))
    n = int(A.value_offsets()[-1])
    A.vals = rng.uniform(0.5, 1, n) * rng.choice([-1.0, 1.0], n)
    if cplx:
        A.vals = A.vals + 1j * rng.uniform(0.5, 1, n) * rng.choice([-1.0, 1.0], n)
    return A


def product(D, stored, X, at):
    """D @ X over the stored elements, X[at[v], v] = +inf (its entry of X is 0)."""
    ref = D @ X
    for v, j in enumerate(at):
        hit = stored[:, j]
        ref.real[hit, v] = np.copysign(np.inf, D[hit, j].real)
        if np.iscomplexobj(ref):
            ref.imag[hit, v] = np.copysign(np.inf, D[hit, j].imag)
    return ref


def agrees(got, ref, tol):
    for g, r in ((got.real, ref.real), (got.imag, ref.imag)):
        fin = np.isfinite(r)
        if not np.array_equal(g[~fin], r[~fin]):
            return False
        if np.abs(np.where(fin, g, 0) - np.where(fin, r, 0)).max() > tol * max(1.0, np.abs(r[fin]).max(initial=0)):
            return False
    return True


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("kind", list(KINDS))
def test_products_and_adjoints(kind, cplx):
    import scipy.sparse as sp
    import torch
    from vbcsr_amd import VBCSR

    A = build(kind, cplx)
    H = VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals)
    if A.n > 4000:  # too wide for a dense copy
        b = KINDS[kind][0][0]
        D = sp.bsr_matrix((A.vals.reshape(-1, b, b), A.col_ind, A.row_ptr), shape=(A.n, A.n)).tocsr()
        stored = None
    else:
        D = A.to_dense()
        stored = D != 0
    rng = np.random.default_rng(5)
    bad = []
    for K in (1, 2, 3, 4, 5, 9, 12, 13, 17, 24, 33, 70) if stored is not None else (1,):
        X = rng.standard_normal((A.n, K)) + (1j * rng.standard_normal((A.n, K)) if cplx else 0.0)
        at = rng.permutation(A.n)[:K] if K <= A.n else rng.integers(0, A.n, K)
        X[at, np.arange(K)] = 0.0
        for adjoint in (False, True):
            M = D.conj().T if adjoint else D
            if stored is None:
                ref = M @ X
                c = M[:, at[0]].toarray().ravel()
                hit = c != 0
                ref.real[hit, 0] = np.copysign(np.inf, c[hit].real)
                if cplx:
                    ref.imag[hit, 0] = np.copysign(np.inf, c[hit].imag)
            else:
                ref = product(M, stored.T if adjoint else stored, X, at)
            for prec in (0, 1, 2):
                if prec == 2 and (adjoint or K > 64):
                    continue
                low = prec == 1
                dt = (np.complex64 if low else np.complex128) if cplx else (np.float32 if low else np.float64)
                xh = X.astype(dt)
                xh[at, np.arange(K)] = np.inf
                x = torch.as_tensor(xh, device="cuda")
                y = torch.full_like(x, 7.0)
                H._core.spmm_raw(K, x.data_ptr(), K, y.data_ptr(), K, prec, adjoint)
                torch.cuda.synchronize()
                if not agrees(y.cpu().numpy(), ref, 1e-12 if prec == 0 else 2e-6):
                    bad.append((K, "adjoint" if adjoint else "forward", prec))
    assert not bad


@pytest.mark.parametrize("kind", ["quads", "mixed"])
@pytest.mark.parametrize("K,nterms", [(1, 1), (1, 3), (3, 1), (2, 35), (5, 13)])
def test_sampled_outer_products(kind, K, nterms):
    """An infinity in the last contraction entry, on real matrices."""
    import torch
    from vbcsr_amd import VBCSR
    from vbcsr_amd.autograd import _lib

    A = build(kind, False)
    H = VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals)
    rng = np.random.default_rng(K + nterms)
    U, V = (rng.uniform(0.5, 1, (nterms, A.n, K)) for _ in range(2))
    V[nterms - 1, :, K - 1] = np.inf
    Ud, Vd = (torch.as_tensor(v, device="cuda") for v in (U, V))
    G = torch.zeros(A.nnz, dtype=torch.float64, device="cuda")
    alpha = np.array([1.0, 0.0])
    p = [ctypes.c_void_p(t.data_ptr()) for t in (Ud, Vd, G)]
    assert _lib().vbh_sddmm_terms(ctypes.c_void_p(H._core.handle), K, nterms, p[0], A.n * K, p[1], A.n * K, 0.5,
                                  alpha.ctypes.data_as(ctypes.c_void_p), p[2], 0, None) == 0
    torch.cuda.synchronize()
    assert np.isposinf(G.cpu().numpy()).all()
