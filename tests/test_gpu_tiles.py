"""Variable-block products and their adjoints at the edges of their kernel:
block sizes around the 4-, 8- and 16-row shapes and above, rows without blocks,
rows of more than 64 slots and of more chunks than one LDS list holds, and
column counts around the lane groups and slices (including more than 64), in
every storage precision, against the oracle.

Tolerances: every sum runs in FP64 over at most about 4000 products of values
of order one, so FP64 results agree to 1e-12 of the largest entry; FP32 storage
rounds matrix values, X entries and results once each (6e-8), so 2e-6."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu

SHAPES = {
    "one": ([1], 40, [0, 1, 3, 17]),
    "edges": ([3, 4, 5, 7, 8, 9], 61, [0, 2, 7, 30]),
    "sixteens": ([15, 16, 17], 33, [1, 5, 33]),
    "mixed": ([1, 4, 9, 13], 90, [0, 4, 70, 90]),
    "up_to_8": ([1, 2, 5, 8], 80, [0, 1, 40, 80]),
    "up_to_8_short": ([1, 2, 5, 8], 80, [0, 1, 3, 9]),  # short rows: the LDS SpMV with one column
    "long_lists": ([2, 33, 21], 75, [75, 3]),  # up to 75 blocks of 6-9 chunks a row
    "widest": ([255, 2, 70], 6, [6, 2]),
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
    for K in (1, 2, 4, 5, 9, 12, 13, 16, 17, 24, 25, 33, 64, 65, 100):
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


@pytest.mark.parametrize("name", ["edges", "mixed", "sixteens", "up_to_8"])
def test_kpm_and_series(name):
    """The fused steps with dots, and the series accumulated in the launch."""
    from vbcsr_amd import VBCSR, kpm
    from vbcsr_amd import workloads as W

    sizes, nb, _ = SHAPES[name]
    rng = np.random.default_rng(2)
    bs = rng.permutation(np.resize(np.array(sizes, np.int32), nb))
    iu, ju, _ = W.random_geometric_pairs(nb, 9.0, rng)
    A = W.scale_to_unit(W.symmetric_from_upper(bs, iu, ju, lambda g, n, r, c, sel: g.standard_normal((n, r, c)), rng))
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
