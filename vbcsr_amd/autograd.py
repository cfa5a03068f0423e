"""Differentiable Chebyshev propagation: psi(T) = U^nsteps psi0 with
U = exp(-i H dt) as a Chebyshev series, as a torch.autograd.Function whose
backward is hand-written on the HIP library (no dense matrices, no torch
autograd through the sparse product).

The forward follows the reference propagator (examples/ex09_graphene_dynamics.py
:102-133, vbcsr/utils.py:71-126): H~ = (H - center) / half_width,
exp(-i H dt) = exp(-i center dt) * sum_n c_n T_n(H~), c_n = (2 - d_n0)
(-i)^n J_n(half_width dt).  The gradient with respect to the stored block values
and to psi0 uses:

* checkpointed recomputation -- psi is kept every ``checkpoint`` steps, and each
  segment is recomputed once during the backward pass;
* per step, the Chebyshev basis t_n (vbh_cheb_basis_terms, which also yields the
  step's result, so a segment's recomputation leaves the bases of its last
  steps behind while they fit a share of the free memory), the Clenshaw
  recurrence with H~^H for the cotangents b_n (vbh_cheb_adjoint_terms), and the
  block-sampled outer products sum_n w_n b_n t_{n-1}^H (vbh_sddmm_terms).

Gradients follow torch's complex convention (dL/dRe + i dL/dIm)."""
from __future__ import annotations

import ctypes
import os
from typing import Optional

import numpy as np
import torch

from . import _core  # noqa: F401  (loads the library with torch's HIP runtime)

_LIB = None


def _lib():
    global _LIB
    if _LIB is None:
        L = ctypes.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "libvbcsr_hip.so"))
        vp, i, d, i64 = ctypes.c_void_p, ctypes.c_int, ctypes.c_double, ctypes.c_int64
        L.vbh_last_error.restype = ctypes.c_char_p
        L.vbh_matrix_set_values.argtypes = [vp, vp, i, vp]
        L.vbh_cheb_apply.argtypes = [vp, i, vp, i, vp, i, i, vp, d, d, i, vp]
        L.vbh_cheb_basis.argtypes = [vp, i, vp, i, i, vp, i, d, d, i, vp]
        L.vbh_cheb_adjoint.argtypes = [vp, i, vp, i, i, vp, vp, i, d, d, i, vp]
        L.vbh_sddmm.argtypes = [vp, i, vp, i, vp, i, vp, vp, i, vp]
        L.vbh_cheb_basis_terms.argtypes = [vp, i, vp, i, i, vp, i64, vp, vp, i, d, d, i, vp]
        L.vbh_cheb_adjoint_terms.argtypes = [vp, i, vp, i, i, vp, vp, i64, d, d, i, vp]
        L.vbh_sddmm_terms.argtypes = [vp, i, i, vp, i64, vp, i64, d, vp, vp, i, vp]
        _LIB = L
    return _LIB


def _check(rc, what):
    if rc != 0:
        raise RuntimeError(f"{what}: {_lib().vbh_last_error().decode()}")


def propagator_coefficients(dt: float, center: float, half_width: float, nterms: int) -> np.ndarray:
    """exp(-i H dt) = sum_n c_n T_n(H~), phase exp(-i center dt) folded into c_n."""
    from scipy.special import jv

    n = np.arange(nterms)
    c = (2.0 - (n == 0)) * (-1j) ** n * jv(n, half_width * dt)
    return (np.exp(-1j * center * dt) * c).astype(np.complex128)


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


class _Ctx:
    """Matrix handle, series and buffers shared by forward and backward."""

    def __init__(self, H, K, nterms, coef, center, half, precision):
        self.H = H
        self.K = K
        self.nterms = nterms
        self.coef = np.ascontiguousarray(coef.view(np.float64))
        self.center = float(center)
        self.half = float(half)
        self.precision = precision
        self.cdtype = torch.complex128 if precision == 0 else torch.complex64

    def load(self, values: torch.Tensor):
        h = self.H._core.handle
        _check(_lib().vbh_matrix_set_values(ctypes.c_void_p(h), ctypes.c_void_p(values.data_ptr()), 1, _stream()),
               "set_values")
        self.H._core.mark_values_written()

    def step(self, psi: torch.Tensor) -> torch.Tensor:
        out = torch.empty_like(psi)
        h = self.H._core.handle
        cp = self.coef.ctypes.data_as(ctypes.c_void_p)
        _check(_lib().vbh_cheb_apply(ctypes.c_void_p(h), self.K, ctypes.c_void_p(psi.data_ptr()), self.K,
                                     ctypes.c_void_p(out.data_ptr()), self.K, self.nterms, cp, self.center,
                                     self.half, self.precision, _stream()), "cheb_apply")
        return out

    def basis(self, psi: torch.Tensor, advance: bool):
        """The step's Chebyshev basis (nterms x N x K) and, with ``advance``, its result."""
        N, K, nt = psi.shape[0], self.K, self.nterms
        T = torch.empty((nt, N, K), dtype=self.cdtype, device=psi.device)
        out = torch.empty_like(psi) if advance else None
        cp = self.coef.ctypes.data_as(ctypes.c_void_p)
        _check(_lib().vbh_cheb_basis_terms(ctypes.c_void_p(self.H._core.handle), K, ctypes.c_void_p(psi.data_ptr()), K,
                                           nt, ctypes.c_void_p(T.data_ptr()), N * K, cp,
                                           ctypes.c_void_p(out.data_ptr()) if advance else None, K, self.center,
                                           self.half, self.precision, _stream()), "cheb_basis_terms")
        return T, out

    def basis_bytes(self, psi: torch.Tensor) -> int:
        return self.nterms * psi.numel() * psi.element_size()

    def step_backward(self, T: torch.Tensor, lam: torch.Tensor, G: torch.Tensor) -> torch.Tensor:
        """Accumulate dL/dvalues of one step (basis T) into G; return dL/dpsi."""
        nt, N, K = T.shape
        L = _lib()
        h = ctypes.c_void_p(self.H._core.handle)
        s = _stream()
        B = torch.empty_like(T)
        cp = self.coef.ctypes.data_as(ctypes.c_void_p)
        _check(L.vbh_cheb_adjoint_terms(h, K, ctypes.c_void_p(lam.data_ptr()), K, nt, cp, ctypes.c_void_p(B.data_ptr()),
                                        N * K, self.center, self.half, self.precision, s), "cheb_adjoint_terms")
        if nt >= 2:  # b_1 t_0^H + 2 sum_{n>=2} b_n t_{n-1}^H
            two = np.array([2.0, 0.0])
            _check(L.vbh_sddmm_terms(h, K, nt - 1, ctypes.c_void_p(B[1:].data_ptr()), N * K,
                                     ctypes.c_void_p(T.data_ptr()), N * K, 0.5, two.ctypes.data_as(ctypes.c_void_p),
                                     ctypes.c_void_p(G.data_ptr()), self.precision, s), "sddmm_terms")
        return B[0].clone()


class ChebPropagation(torch.autograd.Function):
    """psi(T) = [exp(-i H dt)]^nsteps psi0 with H's stored block values taken
    from ``values`` (complex128, slot order, length nnz)."""

    @staticmethod
    def forward(ctx, values, psi0, H, dt, nsteps, nterms, center, half_width, checkpoint, precision):
        coef = propagator_coefficients(dt, center, half_width, nterms)
        c = _Ctx(H, psi0.shape[1], nterms, coef, center, half_width, precision)
        c.load(values)
        psi = psi0.contiguous()
        ckpt = {0: psi}
        for s in range(nsteps):
            psi = c.step(psi)
            if (s + 1) % checkpoint == 0 and s + 1 < nsteps:
                ckpt[s + 1] = psi
        ctx.c = c
        ctx.ckpt = ckpt
        ctx.nsteps = nsteps
        ctx.checkpoint = checkpoint
        ctx.save_for_backward(values)
        return psi

    @staticmethod
    def backward(ctx, grad_out):
        (values,) = ctx.saved_tensors
        c = ctx.c
        c.load(values)  # the matrix may have been changed since the forward pass
        lam = grad_out.to(c.cdtype).contiguous()
        G = torch.zeros(values.shape[0], dtype=torch.complex128, device=values.device)
        starts = sorted(ctx.ckpt)
        for si in range(len(starts) - 1, -1, -1):
            s0 = starts[si]
            s1 = starts[si + 1] if si + 1 < len(starts) else ctx.nsteps
            # recompute the segment's states; its last steps leave their bases,
            # as many as fit an eighth of the free memory (at least the last)
            seg = [ctx.ckpt[s0]]
            keep = max(1, int(torch.cuda.mem_get_info(lam.device)[0] // 8 // max(1, c.basis_bytes(seg[0]))))
            bases = {}
            for k in range(s0, s1):
                last = k == s1 - 1
                if s1 - k <= keep:
                    bases[k], nxt = c.basis(seg[-1], advance=not last)
                else:
                    nxt = c.step(seg[-1])
                if not last:
                    seg.append(nxt)
            for k in range(s1 - 1, s0 - 1, -1):
                T = bases.pop(k) if k in bases else c.basis(seg[k - s0], advance=False)[0]
                lam = c.step_backward(T, lam, G)
                del T
        grad_values = G / c.half
        return grad_values, lam, None, None, None, None, None, None, None, None


def propagate(H, values: torch.Tensor, psi0: torch.Tensor, dt: float, nsteps: int, nterms: int,
              center: float = 0.0, half_width: float = 1.0, checkpoint: int = 10,
              precision: str = "fp64") -> torch.Tensor:
    """Differentiable psi(T) for a complex VBCSR ``H`` (the pattern; values
    come from ``values``).  psi0: (N,) or (N, K) device tensor, complex128 for
    precision "fp64", complex64 for "fp32"."""
    if not H.dtype == np.complex128:
        raise TypeError("propagate needs a complex (complex128) matrix")
    prec = {"fp64": 0, "fp32": 1}[precision]
    want = torch.complex128 if prec == 0 else torch.complex64
    if psi0.dtype != want:
        raise TypeError(f"psi0 must be {want} for precision {precision}")
    if values.dtype != torch.complex128:
        raise TypeError("values must be complex128 (the matrix's storage type)")
    squeeze = psi0.dim() == 1
    p = psi0.reshape(psi0.shape[0], -1)
    out = ChebPropagation.apply(values, p, H, float(dt), int(nsteps), int(nterms), float(center),
                                float(half_width), int(checkpoint), prec)
    return out.reshape(psi0.shape[0]) if squeeze else out
