"""Filled products of filled factors: the dense-panel numeric kernel with a skip
threshold that drops pairs and a filter that drops blocks, against the oracle
(pattern, values, and the count of numeric pairs).  The factors' block norms
span six decades; each case asserts that the kernel's own rule holds (result
filled to 0.8, multiplication paths at least a quarter of all block triples)
and that pairs are skipped and blocks filtered.

Tolerances: at most 60 x 8 products a value; FP64 1e-12 of the largest entry as
elsewhere, FP32 inputs rounded to 2^-24 and a random walk of 480 roundings,
sqrt(480) x 2^-24 = 1.3e-6: 1e-5.  No block norm of the product with the skip
rule lies within 1e-5 of the threshold (asserted), so the patterns agree."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr
from test_gpu_spgemm import _numeric_pairs

pytestmark = pytest.mark.gpu

THR = 0.01


def factor(nb, share, seed):
    """nb block rows of sizes 1..8, each with `share` of the blocks, norms over six decades."""
    from vbcsr_amd import workloads as W

    g = np.random.default_rng(seed)
    bs = g.integers(1, 9, nb).astype(np.int32)
    n = int(np.ceil(share * nb))
    ci = np.concatenate([np.sort(g.choice(nb, n, replace=False)) for _ in range(nb)]).astype(np.int32)
    sizes = bs[np.repeat(np.arange(nb), n)].astype(np.int64) * bs[ci]
    scale = np.repeat(10.0 ** g.uniform(-6, 0, len(ci)), sizes)
    return W.BlockCSR(bs, np.arange(nb + 1) * n, ci, g.standard_normal(int(sizes.sum())) * scale)


def block_norms(M):
    """Norms of the blocks of M M under the skip rule, before the filter."""
    nb, n = M.nb, int(M.row_ptr[1])
    off = np.concatenate([[0], np.cumsum(M.bs)])
    D = M.to_dense()
    blk = [[D[off[i]:off[i + 1], off[j]:off[j + 1]] for j in range(nb)] for i in range(nb)]
    nrm = np.array([[np.linalg.norm(b) for b in row] for row in blk])
    out = []
    for i in range(nb):
        for j in range(nb):
            ks = [k for k in range(nb) if nrm[i, k] > 0 and nrm[k, j] > 0 and not nrm[i, k] * nrm[k, j] < THR / n]
            out.append(np.linalg.norm(sum((blk[i][k] @ blk[k][j] for k in ks), np.zeros((M.bs[i], M.bs[j])))))
    return np.array(out)


@pytest.mark.parametrize("numeric,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
@pytest.mark.parametrize("nb,share", [(17, 0.8), (40, 0.75), (60, 0.7)])
def test_skips_and_filter(nb, share, numeric, tol):
    from vbcsr_amd import VBCSR

    M = factor(nb, share, nb)
    norms = block_norms(M)
    assert np.abs(norms / THR - 1).min() > 1e-5
    H = VBCSR.from_block_csr(M.bs, M.row_ptr, M.col_ind, M.vals)
    C = H.spmm(H, THR, numeric=numeric)
    paths, pairs, before, after = H.spmm_stats
    assert before >= 0.8 * nb * nb and paths >= 0.25 * nb**3  # the panel kernel's rule
    assert pairs < 0.9 * paths and after < before  # pairs skipped, blocks filtered
    ref = O.spgemm(O.Mat.of(M), O.Mat.of(M), THR)
    assert np.array_equal(C.row_ptr, ref.row_ptr) and np.array_equal(C.col_ind, ref.col_ind)
    assert relerr(C.get_values(), ref.vals) < tol
    # pairs whose norms the device rounds to the other side of the threshold: none expected, one allowed per 1000
    want = _numeric_pairs(M, THR)
    assert abs(pairs - want) <= 1e-3 * want, (pairs, want)
