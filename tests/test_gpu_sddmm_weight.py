"""The weight of the first term in the sampled outer products is applied in
FP64 on every block size, also to FP32 vectors: a product of two FP32 entries
is exact in FP64, so sums of at most 18 of them agree with numpy in FP64 to
1e-14 of the largest."""
import ctypes

import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("sizes", [[4], [1, 4, 9]])
@pytest.mark.parametrize("K,nterms", [(1, 1), (1, 3), (3, 6), (5, 2), (9, 2)])
def test_first_weight(sizes, K, nterms, cplx):
    import torch
    from vbcsr_amd import VBCSR
    from vbcsr_amd.autograd import _lib

    rng = np.random.default_rng(K)
    nb = 13
    bs = np.resize(np.array(sizes, np.int32), nb)
    off = np.concatenate([[0], np.cumsum(bs)])
    n = int(off[-1])
    lens = [0, 1, 4, 5, 9]
    cols = [np.sort(rng.choice(nb, lens[i % 5], replace=False)) for i in range(nb)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    nnz = int(sum(bs[i] * bs[c].sum() for i, c in enumerate(cols)))
    H = VBCSR.from_block_csr(bs, rp, np.concatenate(cols).astype(np.int32),
                             np.ones(nnz, complex if cplx else float))
    dt, wide = (np.complex64, np.complex128) if cplx else (np.float32, np.float64)

    def vectors():
        v = rng.standard_normal((nterms, n, K)) + (1j * rng.standard_normal((nterms, n, K)) if cplx else 0.0)
        return v.astype(dt)

    U, V = vectors(), vectors()
    Ud, Vd = (torch.as_tensor(v, device="cuda") for v in (U, V))
    G = torch.zeros(nnz, dtype=getattr(torch, np.dtype(wide).name), device="cuda")
    alpha, first = np.array([2.0, 0.0]), 1.0 / 3.0
    p = [ctypes.c_void_p(t.data_ptr()) for t in (Ud, Vd, G)]
    assert _lib().vbh_sddmm_terms(ctypes.c_void_p(H._core.handle), K, nterms, p[0], n * K, p[1], n * K, first,
                                  alpha.ctypes.data_as(ctypes.c_void_p), p[2], 1, None) == 0
    torch.cuda.synchronize()
    full = sum((first if t == 0 else 1.0) * (U[t].astype(wide) @ V[t].astype(wide).conj().T) for t in range(nterms))
    ref = np.concatenate([2.0 * full[off[i]:off[i + 1], off[j]:off[j + 1]].ravel() for i in range(nb) for j in cols[i]])
    assert relerr(G.cpu().numpy(), ref) < 1e-14
