"""Few block rows with long sums: products whose work-groups share a unit's blocks
between their waves, and blocks of more than 16 rows dealt to several waves, on both
sides of the rules that choose them (block rows x column slices against 512 and 1024
units, one pass of 16 slots, 16 rows a part): rows of more slots and chunks than one
list, empty rows, rows shorter than the waves, in every storage precision, forward and
adjoint, fused steps with dots and series, against the oracle.

Tolerances: every sum runs in FP64 over at most about 20,000 products of values of
order one, so FP64 results agree to 1e-12 of the largest entry; FP32 storage rounds
matrix values, X entries and results once each (6e-8), so 2e-6; moments and series
1e-11, in FP32 2e-5, as elsewhere."""
import numpy as np
import pytest

import oracle as O
import test_gpu_nonfinite as N
from conftest import relerr
from test_gpu_edges_more import symmetric

pytestmark = pytest.mark.gpu

SHAPES = {
    "quads_below": ([4], 4092, [1, 17, 0, 40]),  # 1023 units of one slice
    "quads_above": ([4], 4101, [1, 17, 0, 40]),
    "quads_one_pass": ([4], 39, [16, 3]),
    "quads_few": ([4], 131, [131, 0, 64, 65]),
    "shared": ([1, 4, 9, 13], 130, [0, 3, 130, 70]),
    "not_shared": ([1, 4, 9, 13], 520, [0, 4, 300]),
    "narrow": ([3], 127, [20, 127]),
    "wide_one": ([255], 1, [1]),
    "wide_few": ([255, 2, 70, 16, 17], 7, [7, 2]),
    "wide_some": ([20, 40, 3], 130, [9, 0, 3]),
    "wide_many": ([33, 2, 21], 610, [70, 3]),
}


def build(name, cplx):
    from vbcsr_amd.workloads import BlockCSR

    sizes, nb, lens = SHAPES[name]
    rng = np.random.default_rng(len(name))
    bs = rng.permutation(np.resize(np.array(sizes, np.int32), nb))
    cols = [np.sort(rng.choice(nb, size=min(lens[i % len(lens)], nb), replace=False)) for i in range(nb)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    A = BlockCSR(bs, rp, np.concatenate(cols).astype(np.int32), np.zeros(0))
    n = int(A.value_offsets()[-1])
    A.vals = rng.uniform(-1, 1, n) + (1j * rng.uniform(-1, 1, n) if cplx else 0.0)
    return A


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("name", list(SHAPES))
def test_products_and_adjoints(name, cplx):
    import torch
    from vbcsr_amd import VBCSR

    A = build(name, cplx)
    H, m = VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals), O.Mat.of(A)
    rng = np.random.default_rng(5)
    for K in (1, 2, 13, 24, 33) if A.nb < 1000 else (1, 3, 17):
        X = rng.standard_normal((A.n, K)) + (1j * rng.standard_normal((A.n, K)) if cplx else 0.0)
        for adjoint in (False, True):
            ref = O.spmm_adjoint(m, X) if adjoint else O.spmm(m, X)
            for prec in (0, 1) if adjoint else (0, 1, 2):
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


@pytest.mark.parametrize("sizes,nb,neighbours", [([4], 4100, 20.0), ([4], 60, 30.0), ([1, 4, 9, 13], 70, 40.0),
                                                 ([40, 3], 24, 8.0), ([3], 50, 40.0)])
def test_kpm_and_series(sizes, nb, neighbours):
    from vbcsr_amd import VBCSR, kpm
    from vbcsr_amd import workloads as W

    rng = np.random.default_rng(2)
    bs = rng.permutation(np.resize(np.array(sizes, np.int32), nb))
    iu, ju, _ = W.random_geometric_pairs(nb, neighbours, rng)
    A = W.symmetric_from_upper(bs, iu, ju, lambda g, n, r, c, sel: g.standard_normal((n, r, c)), rng)
    A = W.gershgorin_scale(A)
    H, m = VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals), O.Mat.of(A)
    for K in (1, 2, 10, 19) if nb < 1000 else (1, 4):
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


@pytest.mark.parametrize("name", ["not_shared", "wide_some", "narrow"])
def test_infinities(name, monkeypatch):
    monkeypatch.setitem(N.KINDS, name, SHAPES[name])
    N.test_products_and_adjoints(name, False)


@pytest.mark.parametrize("kind", ["quads", "variable", "wide", "many"])
def test_batches(kind):
    """Batches with few units (shared), with blocks over 16 rows (parts), and with
    enough units for neither; matrices of different sizes, a row without blocks."""
    from vbcsr_amd import VBCSR, kpm

    sizes = {"quads": [4], "variable": [1, 4, 9, 13], "wide": [70, 3, 20], "many": [5, 8]}[kind]
    ms = []
    for q, nb in enumerate((1, 9, 33) if kind != "many" else (70, 70, 70, 70, 70, 70, 70, 70)):
        g = np.random.default_rng(q)
        bs = np.resize(np.array(sizes, np.int64), nb)
        keep = np.triu(g.random((nb, nb)) < 0.8)
        keep = keep | keep.T
        if nb > 2:
            keep[1, :] = keep[:, 1] = False
        keep[0, 0] = True
        ms.append(symmetric(bs, keep, q))
    Hs = [VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals) for A in ms]
    for K in (2, 9, 17, 32, 64):
        vs = []
        for H in Hs:
            v = H.create_multivector(K)
            v.set_random(7 + K, normalize=False)
            vs.append(v)
        refs = [O.kpm_moments(O.Mat.of(A), np.asarray(v.to_numpy()), 19, mode=1) for A, v in zip(ms, vs)]
        for prec, tol in (("fp64", 1e-11), ("fp32", 2e-5), ("mixed", 2e-5)):
            for graph in (True, False):
                got = kpm.kpm_moments_batched(Hs, vs, 19, precision=prec, graph=graph)
                for mu, ref in zip(got, refs):
                    assert relerr(mu, ref) < tol, (K, prec, graph)
