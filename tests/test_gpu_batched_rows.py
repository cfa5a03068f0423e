"""Batched KPM steps on the kernels of single matrices: batches of uniform
blocks of size 1 to 4, of variable blocks, of blocks wider than 16 and of mixed
kinds, with matrices of different sizes (one block row, rows without blocks),
real and complex, column counts around the slices, in a graph and without,
against the oracle.

Tolerances: FP64 1e-11 of the first moment as elsewhere; FP32 vectors or values
round to 6e-8 per step and entry, 2e-5 over 19 moments."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr

pytestmark = pytest.mark.gpu

KINDS = {"one": [1], "two": [2], "three": [3], "four": [4], "variable": [1, 4, 9, 13], "wide": [3, 20], "mixed": None}


def matrix(sizes, nb, cplx, seed):
    from vbcsr_amd.workloads import BlockCSR

    rng = np.random.default_rng(seed)
    bs = rng.permutation(np.resize(np.array(sizes, np.int32), nb))
    n = int(bs.sum())
    keep = np.triu(rng.random((nb, nb)) < min(1.0, 6.0 / nb), 1)
    keep = keep | keep.T | (np.eye(nb, dtype=bool) & (rng.random(nb) < 0.8))
    if nb > 2:
        keep[1, :] = keep[:, 1] = False  # a row without blocks
    D = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)
    D = D + D.conj().T
    off = np.concatenate([[0], np.cumsum(bs)])
    mask = np.repeat(np.repeat(keep, bs, 0), bs, 1)
    D = np.where(mask, D, 0.0)
    D /= 1.1 * max(np.abs(np.linalg.eigvalsh(D)).max(), 1e-3)
    rows, cols = np.nonzero(keep)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nb))]).astype(np.int32)
    vals = [D[off[i]:off[i + 1], off[j]:off[j + 1]].ravel() for i, j in zip(rows, cols)]
    return BlockCSR(bs, rp, cols.astype(np.int32), np.concatenate(vals) if vals else np.zeros(0, D.dtype))


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("kind", list(KINDS))
def test_batches(kind, cplx):
    from vbcsr_amd import VBCSR, kpm

    ms = []
    for q, nb in enumerate((1, 5, 33, 70)):
        sizes = KINDS[kind] or ([1], [4], [2, 3], [8])[q]
        ms.append(matrix(sizes, nb, cplx, 10 * q + len(kind)))
    ms = [A for A in ms if len(A.col_ind)]
    Hs = [VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals) for A in ms]
    for K in (2, 3, 9, 16, 17, 32, 64):
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
