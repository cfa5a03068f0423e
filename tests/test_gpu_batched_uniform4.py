"""A uniform 4 x 4 matrix beside variable ones in a batch: with FP32 values and
32 or 64 columns its block rows run on the block-row wave kernel like all others,
and with a pinned threshold of 1 they belong to the class rows.  Rows without
blocks, one block row, more rows than a work-group; against the oracle.

Tolerances: FP32 vectors or values round to 6e-8 per step and entry, 2e-5 over
19 moments; FP64 1e-11 of the first moment."""
import numpy as np
import pytest

import oracle as O
from conftest import relerr
from test_gpu_batched_rows import matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 64])
@pytest.mark.parametrize("nb4", [1, 5, 70])
def test_beside_variable(nb4, K):
    from vbcsr_amd import VBCSR, kpm

    ms = [matrix([1, 4, 9, 13], 33, False, 1), matrix([4], nb4, False, 5), matrix([8], 6, False, 3)]
    ms = [A for A in ms if len(A.col_ind)]
    Hs = [VBCSR.from_block_csr(A.bs, A.row_ptr, A.col_ind, A.vals) for A in ms]
    vs = []
    for H in Hs:
        v = H.create_multivector(K)
        v.set_random(7 + K, normalize=False)
        vs.append(v)
    refs = [O.kpm_moments(O.Mat.of(A), np.asarray(v.to_numpy()), 19, mode=1) for A, v in zip(ms, vs)]
    try:
        for threshold in (0, 1, -1):
            for prec, tol in (("fp64", 1e-11), ("fp32", 2e-5), ("mixed", 2e-5)):
                kpm.set_batch_plan(threshold)
                got = kpm.kpm_moments_batched(Hs, vs, 19, precision=prec)
                if threshold == 0 and prec != "fp64":
                    assert kpm.last_plan()[0] == -1
                for mu, ref in zip(got, refs):
                    assert relerr(mu, ref) < tol, (threshold, prec)
    finally:
        kpm.set_batch_plan(0)
