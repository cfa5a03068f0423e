"""Column dot products: one block and many, rows around the blocks' shares,
column counts around the threads of a block (more than 256 too), every type,
and calls after one another (the ticket starts over), against FP64 on the host.

Tolerance: a sum of n products of values of order one in FP64, n x 2^-53 of the
sum of their magnitudes with n <= 70,000: 1e-11."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("rows", [1, 255, 256, 257, 1024, 70001])
def test_bdot(rows, cplx):
    from vbcsr_amd import VBCSR

    n = rows
    H = VBCSR.from_block_csr(np.ones(n, np.int32), np.arange(n + 1), np.arange(n, dtype=np.int32),
                             np.ones(n) * (1 + 0j if cplx else 1.0))
    rng = np.random.default_rng(rows)
    for K in (1, 2, 3, 10, 64, 65, 256, 257) if rows < 70000 else (1, 10, 33):
        a, b = H.create_multivector(K), H.create_multivector(K)
        x = rng.standard_normal((n, K)) + (1j * rng.standard_normal((n, K)) if cplx else 0.0)
        y = rng.standard_normal((n, K)) + (1j * rng.standard_normal((n, K)) if cplx else 0.0)
        a.from_numpy(x)
        b.from_numpy(y)
        for p, q, u, w in ((a, b, x, y), (b, a, y, x), (a, a, x, x)):
            ref = (u.conj() * w).sum(0)
            got = np.asarray(p.bdot(q))
            assert np.abs(got - ref).max() <= 1e-11 * np.abs(u.conj() * w).sum(0).max(), (K, rows)
