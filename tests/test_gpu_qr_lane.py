"""GPU: the narrow bands' QR kernels (l <= 7) at the edges of their range:
lengths around their unrolled blocks, tall and wide matrices, the widest upper
band 64 lanes hold and one more, right-hand sides around a wave.  FP64 factors
against the oracle bit for bit; Q'B against the oracle to 1e-13 (its dot
products are summed in pairs); FP32 by Q'A = R to 60 eps of the largest entry
(n reflectors of l+1 <= 8 rows, each off by a few eps of what it touches)."""
import numpy as np
import pytest

from _util import band, bits_equal

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (2, 1), (1, 3), (3, 3), (9, 9), (13, 12), (16, 16), (17, 16), (24, 40), (63, 63), (64, 64), (65, 65),
          (130, 100), (100, 130), (257, 256), (1003, 1000)]


@pytest.mark.parametrize("l,u", [(1, 0), (1, 3), (2, 2), (3, 4), (4, 4), (5, 1), (6, 9), (7, 7), (4, 50), (4, 51), (7, 41), (7, 42)])
def test_factor_and_apply(bh, oracle, l, u):
    for m, n in SHAPES:
        print(f"qr ({l},{u}) {m} x {n}", flush=True)
        rng = np.random.default_rng(m + 7 * n + 31 * l + u)
        A = band(rng, l, u, n, np.float64, dist="n", m=m)
        if n > 20:
            A[:, n // 2] = 0  # a zero column (its reflector may be trivial)
        D, tau = oracle.gbqrf(m, n, l, l + u, oracle.pad_for_lu(A, m, n, l, u))
        F = bh.qr(bh.BandedMatrix.from_host(A, m, l, u))
        assert bits_equal(F.factors.host_data(), D)
        assert bits_equal(F.tau.numpy()[: min(m, n)], tau)
        for nrhs in (1, 3, 64, 65, 130):
            B = np.asfortranarray(rng.standard_normal((m, nrhs)))
            got = (F.Q.T @ bh.DeviceArray.from_numpy(B)).numpy()
            want = oracle.gbqr_qtmul(m, n, l, l + u, D, tau, B)
            assert np.abs(got - want).max() <= 1e-13 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("m,n,l,u", [(65, 65, 1, 1), (130, 100, 4, 4), (100, 130, 7, 3), (257, 257, 3, 40)])
def test_single_precision(bh, m, n, l, u):
    rng = np.random.default_rng(m + l)
    A = band(rng, l, u, n, np.float32, dist="n", m=m)
    M = bh.BandedMatrix.from_host(A, m, l, u)
    F = bh.qr(M)
    got = (F.Q.T @ bh.DeviceArray.from_numpy(np.asfortranarray(M.to_dense()))).numpy()
    R = np.zeros((m, n), np.float32)
    R[: min(m, n)] = F.R_dense()
    if m < n:  # the last row's reflector is the identity: R holds what the band stores of it
        got = np.triu(got)
    assert np.abs(got - R).max() <= 60 * np.finfo(np.float32).eps * np.abs(R).max()


@pytest.mark.parametrize("l,u", [(1, 1), (4, 4), (7, 3)])
@pytest.mark.parametrize("low,high", [(-90, -89), (89, 91), (-160, -150), (150, 153), (-120, 120), (-300, -290)])
def test_exponents(bh, oracle, l, u, low, high):
    """Entries whose squares overflow or vanish: a column whose squares sum to zero keeps what the earlier
    reflectors made of it."""
    m = n = 300
    rng = np.random.default_rng(l + 100 * (high + 400))
    A = band(rng, l, u, n, np.float64, dist="n") * 10.0 ** rng.uniform(low, high, (l + u + 1, n))
    A[:, 40] = 0
    A[u, 80] = 0
    with np.errstate(all="ignore"):
        D, tau = oracle.gbqrf(m, n, l, l + u, oracle.pad_for_lu(np.asfortranarray(A), m, n, l, u))
    F = bh.qr(bh.BandedMatrix.from_host(np.asfortranarray(A), m, l, u))
    got, nan = F.factors.host_data(), np.isnan(D)
    assert (np.isnan(got) == nan).all() and bits_equal(np.where(nan, 0, got), np.where(nan, 0, D))
    assert np.array_equal(F.tau.numpy()[:n], tau, equal_nan=True)
