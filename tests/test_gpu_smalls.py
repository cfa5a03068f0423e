"""Products, adjoints, fused KPM steps and series of uniform blocks of size 1 to
3 at the edges of their kernel: rows without blocks, rows around the slot
batches and partitions, few and many block rows, and column counts around the
lane runs and slices (including more than 64), in every storage precision,
against the oracle.

Tolerances: every sum runs in FP64 over at most 300 products of values of order
one, so FP64 results agree to 1e-12 of the largest entry; FP32 storage rounds
matrix values, X entries and results once each (6e-8), so 2e-6."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu


def build(bs, nb, lens, cplx):
    from vbcsr_amd.workloads import BlockCSR

    rng = np.random.default_rng(bs * 1000 + nb)
    cols = [np.sort(rng.choice(nb, size=min(lens[i % len(lens)], nb), replace=False)) for i in range(nb)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    ci = np.concatenate(cols).astype(np.int32)
    vals = rng.uniform(-1, 1, bs * bs * len(ci)) + (1j * rng.uniform(-1, 1, bs * bs * len(ci)) if cplx else 0.0)
    return BlockCSR(np.full(nb, bs, np.int32), rp, ci, vals)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("bs", [1, 2, 3])
@pytest.mark.parametrize("nb,lens", [(1, [1]), (40, [0, 1, 3, 4, 5, 17]), (700, [0, 7, 12]), (90, [90, 70, 0, 31]),
                                     (9000, [3])])
def test_products_and_adjoints(bs, nb, lens, cplx):
    import torch
    from vbcsr_amd import VBCSR

    A = build(bs, nb, lens, cplx)
    H, m = VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals), O.Mat.of(A)
    rng = np.random.default_rng(5)
    for K in (1, 2, 3, 4, 5, 8, 15, 16, 17, 33, 64, 65, 100) if nb < 9000 else (1, 6, 12):
        X = rng.standard_normal((A.n, K)) + (1j * rng.standard_normal((A.n, K)) if cplx else 0.0)
        for adjoint in (False, True):
            ref = O.spmm_adjoint(m, X) if adjoint else O.spmm(m, X)
            for prec in (0, 1, 2):
                if prec == 2 and (adjoint or K > 64):
                    with pytest.raises(Exception):
                        H._core.spmm_raw(K, 16, K, 16, K, prec, adjoint)
                    continue
                low = prec == 1
                dt = (np.complex64 if low else np.complex128) if cplx else (np.float32 if low else np.float64)
                ld = K + (K % 3)
                x = torch.zeros((A.n, ld), dtype=getattr(torch, np.dtype(dt).name), device="cuda")
                x[:, :K] = torch.as_tensor(X.astype(dt), device="cuda")
                y = torch.full_like(x, 7.0)
                H._core.spmm_raw(K, x.data_ptr(), ld, y.data_ptr(), ld, prec, adjoint)
                torch.cuda.synchronize()
                got = y.cpu().numpy()
                assert relerr(got[:, :K], ref) < (1e-12 if prec == 0 else 2e-6), (K, adjoint, prec)
                assert (got[:, K:] == 7.0).all()


@pytest.mark.parametrize("bs,nb", [(1, 90), (2, 61), (3, 700)])
def test_kpm_and_series(bs, nb):
    """The fused steps with dots, and the series accumulated in the launch."""
    from vbcsr_amd import VBCSR, kpm
    from vbcsr_amd import workloads as W

    rng = np.random.default_rng(2)
    sizes = np.full(nb, bs, np.int32)
    iu, ju, _ = W.random_geometric_pairs(nb, 9.0, rng)
    A = W.scale_to_unit(W.symmetric_from_upper(sizes, iu, ju, lambda g, n, r, c, sel: g.standard_normal((n, r, c)), rng))
    H, m = VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals), O.Mat.of(A)
    for K in (1, 2, 6, 10, 19):
        V = H.create_multivector(K)
        V.set_random(5, normalize=False)
        v0 = np.array(V.to_numpy())
        for mode, code in (("one", 1), ("two", 2)):
            ref = O.kpm_moments(m, v0, 17, mode=code)
            for prec, tol in (("fp64", 1e-11), ("fp32", 2e-5), ("mixed", 2e-5)):
                assert relerr(kpm.kpm_moments(H, V, 17, mode=mode, precision=prec), ref) < tol, (K, mode, prec)
        coef = rng.standard_normal(6) + 0j
        y = np.asarray(memoryview(H._core.cheb_apply(V._core, coef, 0.1, 1.3, 0)))
        assert relerr(y, O.cheb_apply(m, v0, coef, 0.1, 1.3)) < 1e-11, K
