"""Reverse-mode rules for the banded hot path (no reference counterpart: the
reference defines no rrule; its transposed solve src/banded/linalg.jl:41-47 is
the adjoint solve reused here).

  solve_pullback(F, x, xbar)  for x = A \\ b:  bbar = A^{-T} xbar,  Abar = -P(bbar x')
  mul_pullback(A, x0, ybar)   for y = A x0:    Abar = P(ybar x0'),   x0bar = A' ybar
  loss_and_grad(A, b, w, x0)  L = w' A^{-1} b + 1/2 ||A x0||^2 and (dL/dA band, dL/db)
P restricts an outer product to A's band (band storage, like A.data).
"""
from __future__ import annotations

import ctypes as C

from . import _lib
from .bandedmatrix import BandedMatrix, DimensionMismatch, _prefix, mul
from .device import DeviceArray
from .lu import BandedLU, ldiv_, lu


def band_outer_(G: BandedMatrix, alpha1, u1, v1, alpha2=0.0, u2=None, v2=None, beta=1.0) -> BandedMatrix:
    """G <- beta G + P(alpha1 u1 v1' + alpha2 u2 v2') on G's band, in place."""
    m, n = G.shape
    p = _prefix(G.dtype)
    _lib.call(f"bh_{p}gb_band_outer", m, n, G.l, G.u, alpha1, u1.ptr if u1 is not None else None,
              v1.ptr if v1 is not None else None, alpha2, u2.ptr if u2 is not None else None,
              v2.ptr if v2 is not None else None, beta, G.data.ptr, G.data.ld)
    return G


def solve_pullback(F: BandedLU, x: DeviceArray, xbar: DeviceArray, bands):
    """Pullback of x = A \\ b (A square with bandwidths `bands`): (Abar, bbar)."""
    bbar = ldiv_(F.transpose(), xbar.copy())
    n = F.shape[0]
    l, u = bands
    Abar = BandedMatrix.zeros((n, n), (l, u), F.factors.dtype)
    band_outer_(Abar, -1.0, bbar, x, beta=0.0)
    return Abar, bbar


def mul_pullback(A: BandedMatrix, x0: DeviceArray, ybar: DeviceArray):
    """Pullback of y = A x0: (Abar, x0bar)."""
    Abar = BandedMatrix.zeros(A.shape, A.bandwidths(), A.dtype)
    band_outer_(Abar, 1.0, ybar, x0, beta=0.0)
    x0bar = DeviceArray((A.shape[1],), A.dtype)
    mul(x0bar, A, ybar, trans="T")
    return Abar, x0bar


def loss_and_grad(A: BandedMatrix, b: DeviceArray, w: DeviceArray, x0: DeviceArray, method: str = "auto"):
    """L = w' A^{-1} b + 1/2 ||A x0||^2 with its gradient: returns (L, dA, db, x).
    method: the two solves' method (ldiv_'s "auto" -- partitioned from n = 4096
    on, whatever the factors --, "exact", which is a little faster where they are
    dominant and far slower where not, or "partitioned").

    Forward: band LU, 'N' solve, gbmv.  Backward: 'T' solve with the same
    factors and pivots, then one fused band kernel
    dA_ij = fma(y0_i, x0_j, -(lambda_i x_j))."""
    n = A.shape[0]
    # L is a number: one right-hand side (a single column counts) and one weight
    # vector; the kernels below take bare pointers and would read column 0 of more
    if b.shape not in ((n,), (n, 1)):
        raise DimensionMismatch(f"b must be one vector of length {n}, has shape {b.shape}")
    if w.shape != (n,) and not (n == 1 and w.shape == (1, 1)):
        raise DimensionMismatch(f"w must be a vector of length {n}, has shape {w.shape}")
    F = lu(A)
    x = ldiv_(F, b.copy(), method)
    y0 = DeviceArray((n,), A.dtype)
    mul(y0, A, x0)
    lam = ldiv_(F.transpose(), w.copy(), method)
    dA = BandedMatrix.zeros((n, n), A.bandwidths(), A.dtype)
    _lib.call(f"bh_{_prefix(A.dtype)}gb_band_grad", n, n, A.l, A.u, lam.ptr, x.ptr, y0.ptr, x0.ptr, dA.data.ptr,
              dA.data.ld)
    L = C.c_double(0.0)
    _lib.call(f"bh_{_prefix(A.dtype)}gb_loss", n, w.ptr, x.ptr, y0.ptr, C.byref(L))
    return L.value, dA, lam, x
