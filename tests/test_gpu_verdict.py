"""GPU: which way a call went that can run by blocks (bh_cut_verdict): the blocks
agreed (1), the gate refused the matrix (2), a seam differed and the sequential
kernels ran (3), no blocks (0).  test_gpu_cut.py compares the bits, which are
the same every way; here each way is shown to be taken."""
import ctypes as C

import numpy as np
import pytest

from _util import band

pytestmark = pytest.mark.gpu

FP = {np.float64: "d", np.float32: "s"}
DTYPES = [np.float64, np.float32]
AGREED, REFUSED, DIFFERED, NONE = 1, 2, 3, 0


def verdict(bh):
    v, t = C.c_int(-1), C.c_int(-1)
    bh._lib.call("bh_cut_verdict", C.byref(v), C.byref(t))
    return v.value, t.value


@pytest.fixture(autouse=True)
def _allowed(monkeypatch):
    monkeypatch.delenv("BANDEDHIP_CUT", raising=False)


def _dominant(n, kl, ku, dtype, shift):
    A = band(np.random.default_rng(n + kl), kl, ku, n, np.float64, dist="n")
    A[ku] += shift
    return np.asfortranarray(A.astype(dtype))


def _gbtrf(bh, A, n, kl, ku):
    """(factors, pivots) on the device and as host arrays."""
    ld = 2 * kl + ku + 1
    ab = np.zeros((ld, n), A.dtype, order="F")
    ab[kl:] = A
    d, p, info = bh.DeviceArray.from_numpy(ab), bh.DeviceArray((n,), np.int64), C.c_int64(-1)
    bh._lib.call(f"bh_{FP[A.dtype.type]}gbtrf", n, n, kl, ku, d.ptr, ld, p.ptr, C.byref(info))
    assert info.value == 0
    return d, p


def _stretch(n, length, dtype, kd=1, off=-1.0, strong=4.0):
    """Second differences whose diagonal is 2 over `length` columns in the middle: there the chain does not forget."""
    A = np.zeros((3, n), order="F")
    A[0], A[2], A[1] = off, off, strong
    m = n // 2
    A[1, m:m + length] = 2
    return np.asfortranarray(A.astype(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,kl,ku", [
    (1000, 1, 1), (10000, 4, 3), (10001, 8, 8), (5000, 16, 3),  # one wave to a block
    (6001, 11, 5), (7000, 15, 16),  # its wider half
    (12000, 40, 50), (9000, 70, 60),  # the blocked kernel
    (16400, 16, 16), (12345, 100, 128),  # the MFMA kernel
])
def test_lu(bh, dtype, n, kl, ku):
    _gbtrf(bh, _dominant(n, kl, ku, dtype, 2 * (kl + ku) + 2), n, kl, ku)
    assert verdict(bh) == (AGREED, 1)
    _gbtrf(bh, _dominant(n, kl, ku, dtype, 0), n, kl, ku)
    assert verdict(bh)[0] == REFUSED


def test_none(bh, monkeypatch):
    A = _dominant(100, 1, 1, np.float64, 9)
    _gbtrf(bh, A, 100, 1, 1)
    assert verdict(bh) == (NONE, 0)  # too short
    monkeypatch.setenv("BANDEDHIP_CUT", "off")
    _gbtrf(bh, _dominant(10000, 1, 1, np.float64, 9), 10000, 1, 1)
    assert verdict(bh) == (NONE, 0)


@pytest.mark.parametrize("dtype", DTYPES)
def test_lu_second_try(bh, monkeypatch, dtype):
    """Blocks that begin in the stretch differ; with four times the lead-in they begin before it.  A system too short
    for a second try goes to the sequential kernel."""
    for n, want in ((20000, (AGREED, 2)), (10000, (DIFFERED, 1))):
        A = _stretch(n, 200, dtype)
        f, p = _gbtrf(bh, A, n, 1, 1)
        assert verdict(bh) == want
        monkeypatch.setenv("BANDEDHIP_CUT", "off")
        f0, p0 = _gbtrf(bh, A, n, 1, 1)
        monkeypatch.delenv("BANDEDHIP_CUT")
        assert f.numpy().tobytes() == f0.numpy().tobytes() and p.numpy().tobytes() == p0.numpy().tobytes()


def test_lu_longer_than_the_whole_kernels_offsets(bh):
    """2 GiB of band storage: the blocks take it, the one-wave kernel for the whole system does not (its byte offsets
    have 32 bits).  The pivots of a constant tridiagonal matrix reach their fixed point within some 30 columns."""
    n, ld = (1 << 26) + 5, 4
    ab = np.empty((ld, n), order="F")
    ab[0], ab[1], ab[2], ab[3] = 0, -1, 4, -1
    d, p, info = bh.DeviceArray.from_numpy(ab), bh.DeviceArray((n,), np.int64), C.c_int64(-1)
    bh._lib.call("bh_dgbtrf", n, n, 1, 1, d.ptr, ld, p.ptr, C.byref(info))
    assert info.value == 0 and verdict(bh) == (AGREED, 1)
    f = d.numpy()
    x = 4.0
    for _ in range(60):
        x = 4.0 - 1.0 / x
    assert np.abs(f[2, 60:] - x).max() <= 4 * np.spacing(x) and np.abs(f[3, 60:-1] + 1 / x).max() <= 4 * np.spacing(1 / x)
    assert (f[1, 1:] == -1).all() and (f[0, 2:] == 0).all()
    assert (p.numpy() == np.arange(1, n + 1)).all()


def _tri(n, k, up, dtype, diag, length=0):
    A = np.random.default_rng(n + k).uniform(-1, 1, (k + 1, n)) * (0.5 / k)
    d = k if up else 0
    A[d] = diag
    if length:  # x_j = b_j + x_{j +- 1}: nothing decays
        m = n // 2
        A[:, m:m + length] = 0
        A[d, m:m + length] = 1
        A[k - 1 if up else 1, m:m + length] = -1
    return np.asfortranarray(A.astype(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("uplo,trans", [("U", "N"), ("L", "N"), ("U", "T"), ("L", "T")])
@pytest.mark.parametrize("n,k,length", [(3000, 1, 400), (20000, 8, 3000), (20031, 16, 3000), (40001, 100, 8000)])
def test_triangular(bh, dtype, uplo, trans, n, k, length):
    x = bh.DeviceArray.from_numpy(np.random.default_rng(1).standard_normal(n).astype(dtype))

    def solve(A):
        d = bh.DeviceArray.from_numpy(A)
        bh._lib.call(f"bh_{FP[dtype]}tbsv", uplo.encode(), trans.encode(), b"N", n, k, d.ptr, k + 1, x.ptr, 1)
        return verdict(bh)

    up = uplo == "U"
    assert solve(_tri(n, k, up, dtype, 1.5)) == (AGREED, 1)
    assert solve(_tri(n, k, up, dtype, 0.1))[0] == REFUSED
    assert solve(_tri(n, k, up, dtype, 1.5, length))[0] == DIFFERED


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("uplo,ldl,n,kd", [("U", False, 1003, 2), ("U", False, 4096, 8), ("U", False, 9001, 17), ("L", False, 4096, 8),
                                           ("L", True, 4096, 8), ("U", True, 12000, 64)])
def test_cholesky(bh, dtype, uplo, ldl, n, kd):
    d = kd if uplo == "U" else 0

    def factor(diag, length=0):
        A = np.random.default_rng(n).uniform(-1, 1, (kd + 1, n))
        A[d] = diag + np.random.default_rng(3).random(n)
        if length:  # second differences there, uncoupled from the rest
            m = n // 2
            A[np.arange(kd + 1) != d, m - kd:m + length + kd] = 0
            A[d, m:m + length] = 2
            A[kd - 1 if uplo == "U" else 1, m:m + length] = -1
        x, info = bh.DeviceArray.from_numpy(np.asfortranarray(A.astype(dtype))), C.c_int64(-1)
        if ldl:
            bh._lib.call(f"bh_{FP[dtype]}sbldlt", uplo.encode(), n, kd, x.ptr, kd + 1)
        else:
            bh._lib.call(f"bh_{FP[dtype]}pbtrf", uplo.encode(), n, kd, x.ptr, kd + 1, C.byref(info))
            assert diag < 1 or info.value == 0
        return verdict(bh)

    assert factor(kd + 1) == (AGREED, 1)
    assert factor(0.2)[0] == REFUSED
    assert factor(kd + 1, n // 6)[0] == DIFFERED


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n,kl,ku,nrhs", [(4097, 4, 4, 3), (20001, 3, 8, 1), (30000, 16, 16, 1), (40000, 128, 128, 1), (6000, 0, 5, 2)])
def test_lu_solve(bh, dtype, trans, n, kl, ku, nrhs):
    b = bh.DeviceArray.from_numpy(np.asfortranarray(np.random.default_rng(1).standard_normal((n, nrhs)).astype(dtype)))
    p, nb = FP[dtype], C.c_size_t(0)
    bh._lib.call("bh_gbtrs_part_workspace", p.encode(), n, kl, ku, nrhs, C.byref(nb))
    for shift, want in ((2 * (kl + ku) + 2, AGREED), (0, REFUSED)):
        f, piv = _gbtrf(bh, _dominant(n, kl, ku, dtype, shift), n, kl, ku)
        args = (n, kl, ku, nrhs, f.ptr, 2 * kl + ku + 1, piv.ptr, b.ptr, n)
        bh._lib.call(f"bh_{p}gbtrs", trans.encode(), *args)
        assert verdict(bh)[0] == want
        if nb.value and (want == AGREED or kl > 0):  # (a random triangle grows past the partitioned solve's bound)
            ws = bh.DeviceArray((nb.value,), np.uint8)
            bh._lib.call(f"bh_{p}gbtrs_part", trans.encode(), *args, ws.ptr, nb.value)
            assert verdict(bh)[0] == want


@pytest.mark.parametrize("dtype", DTYPES)
def test_lu_solve_differs(bh, monkeypatch, dtype):
    """Dominant factors with a stretch that does not forget: every solve takes its fallback, with the bits (partitioned:
    the rounding) of the call without blocks."""
    n = 20000
    f, piv = _gbtrf(bh, _stretch(n, 2000, dtype), n, 1, 1)
    b, p, nb = np.random.default_rng(1).standard_normal(n).astype(dtype), FP[dtype], C.c_size_t(0)
    bh._lib.call("bh_gbtrs_part_workspace", p.encode(), n, 1, 1, 1, C.byref(nb))
    part = bh.DeviceArray((nb.value,), np.uint8)
    bh._lib.call("bh_gbtrs_blocked_workspace", p.encode(), n, 1, 1, C.byref(nb))
    blk = bh.DeviceArray((nb.value,), np.uint8)
    for name, trans, ws in (("gbtrs", "N", None), ("gbtrs", "T", None), ("gbtrs_part", "N", part), ("gbtrs_part", "T", part),
                            ("gbtrs_blocked", None, blk)):
        out = []
        for cut in (True, False):
            if not cut:
                monkeypatch.setenv("BANDEDHIP_CUT", "off")
            x = bh.DeviceArray.from_numpy(b)
            t = [trans.encode()] if trans else []
            w = [ws.ptr, ws.nbytes] if ws is not None else []
            bh._lib.call(f"bh_{p}{name}", *t, n, 1, 1, 1, f.ptr, 4, piv.ptr, x.ptr, n, *w)
            assert verdict(bh)[0] == (DIFFERED if cut else NONE), (name, trans)
            out.append(x.numpy())
            monkeypatch.delenv("BANDEDHIP_CUT", raising=False)
        assert out[0].tobytes() == out[1].tobytes(), (name, trans)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,kl,ku,nrhs", [(6000, 1, 1, 1), (20001, 16, 20, 16), (65536, 128, 128, 3)])
def test_blocked_solve(bh, dtype, n, kl, ku, nrhs):
    b = bh.DeviceArray.from_numpy(np.asfortranarray(np.random.default_rng(1).standard_normal((n, nrhs)).astype(dtype)))
    p, nb = FP[dtype], C.c_size_t(0)
    bh._lib.call("bh_gbtrs_blocked_workspace", p.encode(), n, kl, ku, C.byref(nb))
    ws = bh.DeviceArray((nb.value,), np.uint8)
    for shift, want in ((2 * (kl + ku) + 2, AGREED), (0, REFUSED)):
        f, piv = _gbtrf(bh, _dominant(n, kl, ku, dtype, shift), n, kl, ku)
        bh._lib.call(f"bh_{p}gbtrs_blocked", n, kl, ku, nrhs, f.ptr, 2 * kl + ku + 1, piv.ptr, b.ptr, n, ws.ptr, nb.value)
        assert verdict(bh)[0] == want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("ldl", [False, True])
@pytest.mark.parametrize("n,kd", [(5120, 64), (65536, 8), (20000, 20), (10001, 1), (1999, 1)])
def test_laplacians_are_not_tried(bh, dtype, uplo, ldl, n, kd):
    """The second difference and the five-point Laplacian never forget where a chain began, although their diagonal is
    twice the sum of the stored half: the gate refuses them.  With 16 times the diagonal it does not.  The slots
    outside the matrix hold NaN."""
    up = uplo == "U"
    A = np.zeros((kd + 1, n))
    if kd > 1:
        A[0 if up else kd] = -1
    A[kd - 1 if up else 1] = -1
    if kd > 1:  # a grid's rows are not coupled end to end
        A[kd - 1 if up else 1, (0 if up else kd - 1)::kd] = 0
    for c in range(kd):
        if up:
            A[:kd - c, c] = np.nan
        else:
            A[c + 1:, n - 1 - c] = np.nan
    for scale, want in ((1, REFUSED), (16, AGREED)):
        A[kd if up else 0] = scale * (2 if kd == 1 else 4)
        x, info = bh.DeviceArray.from_numpy(np.asfortranarray(A.astype(dtype))), C.c_int64(0)
        if ldl:
            bh._lib.call(f"bh_{FP[dtype]}sbldlt", uplo.encode(), n, kd, x.ptr, kd + 1)
        else:
            bh._lib.call(f"bh_{FP[dtype]}pbtrf", uplo.encode(), n, kd, x.ptr, kd + 1, C.byref(info))
        assert info.value == 0 and verdict(bh)[0] == want, scale


@pytest.mark.parametrize("uplo,trans", [("U", "N"), ("L", "T")])
def test_impulse(bh, monkeypatch, uplo, trans):
    """A right-hand side that is zero but for one entry: the tail of the solution is what a block among the zeros
    cannot know.  The seams differ and the result is the sequential kernel's."""
    n, k = 20000, 4
    a = bh.DeviceArray.from_numpy(_tri(n, k, uplo == "U", np.float64, 1.5))
    b = np.zeros(n)
    b[n - 5000] = 1
    out = []
    for cut in (True, False):
        if not cut:
            monkeypatch.setenv("BANDEDHIP_CUT", "off")
        x = bh.DeviceArray.from_numpy(b)
        bh._lib.call("bh_dtbsv", uplo.encode(), trans.encode(), b"N", n, k, a.ptr, k + 1, x.ptr, 1)
        assert verdict(bh)[0] == (DIFFERED if cut else NONE)
        out.append(x.numpy())
    assert out[0].tobytes() == out[1].tobytes()
    assert np.count_nonzero(out[0]) > 20 * k + 64 * 2  # a tail longer than the lead-in
