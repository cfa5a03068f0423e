"""FP32 Chebyshev series: every term is added in FP64 with the FP64 coefficient
and rounded to FP32 once, whichever kernel runs the step.  On the identity
t_n = x for every n without rounding, and x has four significant bits, so the
series is reproduced exactly: the results are compared bit by bit (the first
term is a product in the vectors' own type)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = {
    "one": ([1], 60, 3),
    "two": ([2], 61, 2),
    "many_one": ([1], 8192, 1),
    "many_two": ([2], 8193, 2),
    "many_three": ([3], 8200, 2),
    "quads": ([4], 37, 5),
    "variable": ([1, 4, 9, 13], 40, 10),
    "up_to_8": ([1, 3, 5, 8], 50, 10),
    "up_to_8_short": ([1, 3, 5, 8], 50, 3),
}


def identity(kind, cplx):
    """The identity with zero blocks stored beside the diagonal."""
    from vbcsr_amd import VBCSR

    sizes, nb, slots = KINDS[kind]
    bs = np.resize(np.array(sizes, np.int32), nb)
    cols = [np.sort((i + np.arange(slots)) % nb) for i in range(nb)]
    rp = (np.arange(nb + 1) * slots).astype(np.int32)
    parts = [np.eye(bs[i]).ravel() if j == i else np.zeros(bs[i] * bs[j]) for i in range(nb) for j in cols[i]]
    vals = np.concatenate(parts)
    return int(bs.sum()), VBCSR.from_block_csr(bs, rp, np.concatenate(cols).astype(np.int32),
                                               vals.astype(complex) if cplx else vals)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("kind", list(KINDS))
def test_series_rounding(kind, cplx):
    import torch
    from vbcsr_amd.autograd import _lib

    n, H = identity(kind, cplx)
    rng = np.random.default_rng(3)
    nt = 40
    coef = rng.standard_normal(nt) + (1j * rng.standard_normal(nt) if cplx else 0j)
    cp = np.ascontiguousarray(coef).view(np.float64)
    for K in (1, 2, 5):
        # real vectors: the imaginary parts of complex ones stay zero, so every product is exact
        x = (rng.integers(8, 16, (n, K)) / 8.0).astype(np.float32)
        dt = np.complex64 if cplx else np.float32
        xd = torch.as_tensor(x.astype(dt), device="cuda")
        y = torch.zeros_like(xd)
        assert _lib().vbh_cheb_apply(ctypes.c_void_p(H._core.handle), K, ctypes.c_void_p(xd.data_ptr()), K,
                                     ctypes.c_void_p(y.data_ptr()), K, nt, cp.ctypes.data_as(ctypes.c_void_p), 0.0, 1.0,
                                     1, None) == 0
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        for part, c in ((got.real, coef.real), (got.imag, coef.imag)):
            ref = np.float32(c[0]) * x
            for cn in c[1:]:
                ref = (cn * x.astype(np.float64) + ref.astype(np.float64)).astype(np.float32)
            assert np.array_equal(part, ref), (K, np.abs(part - ref).max())
