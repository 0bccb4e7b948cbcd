"""GPU: systems cut into blocks that run at once (csrc/bh_cut.hpp) against the
same entry points with cutting switched off.  Whether a system is cut and its
seams agree, or the sequential kernels run, the outputs are the same bits: the
lead-in's rounding is checked, not trusted.  Inputs that must fall back (weak
diagonals, a zero column, a NaN, interchanges) are mixed with dominant ones,
at sizes around the edges of the blocks."""
import ctypes as C
import threading

import numpy as np
import pytest

from _util import band

pytestmark = pytest.mark.gpu

FP = {np.float64: "d", np.float32: "s"}


def _both(monkeypatch, f):
    """f() with cutting allowed and with it off."""
    monkeypatch.delenv("BANDEDHIP_CUT", raising=False)
    on = f()
    monkeypatch.setenv("BANDEDHIP_CUT", "off")
    off = f()
    return on, off


def _same(on, off):
    for a, b in zip(on, off):
        if isinstance(a, np.ndarray):
            assert a.shape == b.shape and a.tobytes() == b.tobytes(), np.argwhere(a != b)[:5]
        else:
            assert a == b


def _system(rng, n, kl, ku, dtype, kind):
    A = band(rng, kl, ku, n, np.float64, dist="n")
    A[ku, :] += 2 * (kl + ku) + 2
    if kind == "weak":  # a stretch whose diagonal does not dominate: interchanges, and slow or no agreement
        A[ku, n // 3 : n // 3 + 200] -= 2 * (kl + ku) + 2
    elif kind == "zero":
        A[:, n // 2] = 0
    elif kind == "nan":
        A[ku, n // 2] = np.nan
    elif kind == "random":
        A = band(rng, kl, ku, n, np.float64, dist="u")
    return np.asfortranarray(A.astype(dtype))


LU = [  # n, kl, ku: lane kernel, its edges; the MFMA kernel for long and for wide bands
    (1000, 1, 1), (1003, 2, 5), (4096, 4, 4), (10000, 4, 3), (10001, 8, 8), (5000, 16, 3), (16383, 8, 8),
    (16384, 8, 8), (16400, 16, 16), (262144, 9, 9), (30001, 9, 20), (9000, 64, 70), (12345, 100, 128), (3000, 33, 65),
    (5000, 9, 2), (6001, 11, 5), (20000, 13, 3), (7000, 15, 16),  # the lane kernel's wider half
    (5000, 20, 20), (12000, 40, 50), (6000, 16, 50), (9000, 70, 60),  # the blocked kernel
]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["dominant", "weak", "zero", "nan", "random"])
@pytest.mark.parametrize("n,kl,ku", LU)
def test_lu(bh, monkeypatch, dtype, kind, n, kl, ku):
    if kind != "dominant" and n > 12000:
        pytest.skip("the fallbacks are the same code at every length")
    print(f"lu {dtype.__name__} {kind} n={n} ({kl},{ku})", flush=True)
    A = _system(np.random.default_rng(n + kl), n, kl, ku, dtype, kind)
    ld = 2 * kl + ku + 2  # a leading dimension one larger than the band
    ab = np.full((ld, n), 7, dtype, order="F")
    ab[kl : 2 * kl + ku + 1] = A

    def run():
        d = bh.DeviceArray.from_numpy(ab)
        ipiv, info = bh.DeviceArray((n,), np.int64), C.c_int64(-7)
        bh._lib.call(f"bh_{FP[dtype]}gbtrf", n, n, kl, ku, d.ptr, ld, ipiv.ptr, C.byref(info))
        f, p = d.numpy(), ipiv.numpy()
        # pivots and columns past a zero pivot are defined, those past a NaN compare by bits too
        return f, p, info.value

    on, off = _both(monkeypatch, run)
    if kind == "dominant":
        assert off[2] == 0
    _same(on, off)


def _triangle(rng, n, k, up, dtype, kind):
    A = rng.uniform(-1, 1, (k + 1, n)) * (0.5 / max(k, 1))
    d = k if up else 0
    A[d] = 1 + rng.random(n)
    if kind == "weak":
        A[d, n // 3 : n // 3 + 300] = 0.01
    elif kind == "zero":
        A[d, n // 2] = 0
    elif kind == "nan":
        A[(d + 1) % (k + 1), n // 2] = np.nan
    return np.asfortranarray(A.astype(dtype))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo,trans", [("U", "N"), ("L", "N"), ("U", "T"), ("L", "T")])
@pytest.mark.parametrize("kind", ["dominant", "weak", "zero", "nan"])
@pytest.mark.parametrize("n,k,nrhs,incx,diag", [
    (3000, 1, 1, 1, "N"), (4097, 3, 3, 1, "N"), (20000, 8, 1, 2, "U"), (20031, 16, 2, 1, "N"), (30000, 64, 1, 1, "N"),
    (40001, 100, 2, 1, "U"), (66000, 200, 1, 1, "N"), (5000, 0, 1, 1, "N"),
])
def test_triangular(bh, monkeypatch, dtype, uplo, trans, kind, n, k, nrhs, incx, diag):
    if kind == "nan" and k == 0:
        pytest.skip("a diagonal matrix has no chain")
    print(f"tbsv {dtype.__name__} {uplo}{trans}{diag} {kind} n={n} k={k} nrhs={nrhs} incx={incx}", flush=True)
    rng = np.random.default_rng(n + k)
    A = bh.DeviceArray.from_numpy(_triangle(rng, n, k, uplo == "U", dtype, kind))
    b = rng.standard_normal(n * incx if nrhs == 1 else (n + 3, nrhs)).astype(dtype)
    p, u, t, d = FP[dtype], uplo.encode(), trans.encode(), diag.encode()

    def run():
        x = bh.DeviceArray.from_numpy(b)
        if nrhs == 1:
            bh._lib.call(f"bh_{p}tbsv", u, t, d, n, k, A.ptr, A.ld, x.ptr, incx)
        else:
            bh._lib.call(f"bh_{p}tbsv_multi", u, t, d, n, k, A.ptr, A.ld, nrhs, x.ptr, n + 3)
        return (x.numpy(),)

    _same(*_both(monkeypatch, run))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("ldl", [False, True])
@pytest.mark.parametrize("kind", ["dominant", "weak", "zero", "nan"])
@pytest.mark.parametrize("n,kd", [(500, 1), (1003, 2), (4096, 8), (9001, 17), (12000, 64), (30000, 128)])
def test_cholesky(bh, monkeypatch, dtype, uplo, ldl, kind, n, kd):
    if kd > 120 and (dtype == np.float64 or kind != "dominant"):
        pytest.skip("the LDS window holds it in single precision; one long chain is enough")
    print(f"cholesky {dtype.__name__} {uplo} ldl={ldl} {kind} n={n} kd={kd}", flush=True)
    rng = np.random.default_rng(n + kd)
    A = rng.uniform(-1, 1, (kd + 1, n))
    d = kd if uplo == "U" else 0
    A[d] = kd + 2 + rng.random(n)
    if kind == "weak":  # not positive definite there: info > 0, or no agreement
        A[d, n // 3 : n // 3 + 40] = 0.3
    elif kind == "zero":
        A[d, n // 2] = 0
    elif kind == "nan":
        A[d, n // 2] = np.nan
    ab = np.full((kd + 3, n), 5, dtype, order="F")
    ab[: kd + 1] = A

    def run():
        x, info = bh.DeviceArray.from_numpy(ab), C.c_int64(-7)
        if ldl:
            bh._lib.call(f"bh_{FP[dtype]}sbldlt", uplo.encode(), n, kd, x.ptr, kd + 3)
            return x.numpy(), 0
        bh._lib.call(f"bh_{FP[dtype]}pbtrf", uplo.encode(), n, kd, x.ptr, kd + 3, C.byref(info))
        return x.numpy(), info.value

    _same(*_both(monkeypatch, run))


def _swapped(rng, n, kl, ku, dtype):
    """Dominant rows 2i and 2i+1 exchanged: half the steps interchange, and the factors are dominant."""
    A = band(rng, kl - 1, ku - 1, n, np.float64, dist="n")
    A[ku - 1] += 2 * (kl + ku) + 2
    B = np.zeros((kl + ku + 1, n))
    for r in range(kl + ku - 1):  # entry (i, j), i = j + r - (ku - 1), moves to row i ^ 1
        i = np.arange(n) + r - (ku - 1)
        to = np.where((i | 1) < n, i ^ 1, i)
        ok = (i >= 0) & (i < n)
        B[(ku + to - np.arange(n))[ok], np.arange(n)[ok]] = A[r, ok]
    return np.asfortranarray(B.astype(dtype))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("kind", ["dominant", "swapped", "random", "nan"])
@pytest.mark.parametrize("n,kl,ku,nrhs", [
    (2000, 1, 1, 1), (4097, 4, 4, 3), (20001, 8, 3, 1), (20000, 3, 9, 2), (30000, 16, 16, 1), (16385, 40, 30, 1),
    (40000, 128, 128, 1), (6000, 0, 5, 2),
])
def test_lu_solve(bh, monkeypatch, dtype, trans, kind, n, kl, ku, nrhs):
    if kind in ("swapped", "nan") and kl == 0:
        pytest.skip("no interchanges")
    print(f"gbtrs {dtype.__name__} {trans} {kind} n={n} ({kl},{ku}) nrhs={nrhs}", flush=True)
    rng = np.random.default_rng(n + kl)
    A = _swapped(rng, n, kl, ku, dtype) if kind == "swapped" else _system(
        rng, n, kl, ku, dtype, "random" if kind == "random" else "dominant")
    F = bh.lu(bh.BandedMatrix.from_host(A, n, kl, ku))
    if kind == "swapped":
        assert (F.ipiv != np.arange(1, n + 1)).sum() > n // 3
    if kind == "nan":
        f = F.factors.host_data()
        f[kl + ku + 1, n // 2] = np.nan
        F.factors.data.upload(f)
    b = rng.standard_normal((n + 1, nrhs)).astype(dtype)
    p, t = FP[dtype], trans.encode()
    args = (n, kl, ku, nrhs, F.factors.data.ptr, F.factors.data.ld, F.ipiv_dev.ptr)

    def run():
        x = bh.DeviceArray.from_numpy(b)
        bh._lib.call(f"bh_{p}gbtrs", t, *args, x.ptr, n + 1)
        return (x.numpy(),)

    on, off = _both(monkeypatch, run)
    _same(on, off)
    nb = C.c_size_t(0)
    bh._lib.call("bh_gbtrs_part_workspace", p.encode(), n, kl, ku, nrhs, C.byref(nb))
    if nb.value and kind in ("dominant", "swapped"):
        # the partitioned solve takes the blocks too: then its bits are the exact solve's
        monkeypatch.delenv("BANDEDHIP_CUT", raising=False)
        ws, x = bh.DeviceArray((nb.value,), np.uint8), bh.DeviceArray.from_numpy(b)
        bh._lib.call(f"bh_{p}gbtrs_part", t, *args, x.ptr, n + 1, ws.ptr, nb.value)
        got, eps = x.numpy().astype(np.float64), np.finfo(dtype).eps
        # (and where the blocks were refused, rounding: the triangles' condition is under 10 at this dominance)
        assert np.abs(got - off[0]).max() <= 100 * (kl + ku + 1) * eps * np.abs(off[0]).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["dominant", "swapped", "random", "nan"])
@pytest.mark.parametrize("n,kl,ku,nrhs", [(6000, 1, 1, 1), (20001, 16, 20, 16), (30000, 40, 17, 17), (65536, 128, 128, 3)])
def test_blocked_solve(bh, monkeypatch, dtype, kind, n, kl, ku, nrhs):
    print(f"gbtrs_blocked {dtype.__name__} {kind} n={n} ({kl},{ku}) nrhs={nrhs}", flush=True)
    rng = np.random.default_rng(n + kl)
    A = _swapped(rng, n, kl, ku, dtype) if kind == "swapped" else _system(
        rng, n, kl, ku, dtype, "random" if kind == "random" else "dominant")
    F = bh.lu(bh.BandedMatrix.from_host(A, n, kl, ku))
    if kind == "nan":
        f = F.factors.host_data()
        f[kl + ku + 1, n // 2] = np.nan
        F.factors.data.upload(f)
    b, p, nb = rng.standard_normal((n + 5, nrhs)).astype(dtype), FP[dtype], C.c_size_t(0)
    bh._lib.call("bh_gbtrs_blocked_workspace", p.encode(), n, kl, ku, C.byref(nb))
    ws = bh.DeviceArray((nb.value,), np.uint8)

    def run():
        x = bh.DeviceArray.from_numpy(b)
        bh._lib.call(f"bh_{p}gbtrs_blocked", n, kl, ku, nrhs, F.factors.data.ptr, F.factors.data.ld, F.ipiv_dev.ptr,
                     x.ptr, n + 5, ws.ptr, nb.value)
        return (x.numpy(),)

    _same(*_both(monkeypatch, run))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kd", range(1, 10))
def test_cholesky_narrow(bh, monkeypatch, dtype, kd):
    """Every width of the one-lane-per-block kernel and one more, at lengths around its blocks; NaN in the unused corner."""
    for n in (600, 601, 1999, 8192, 20011):
        print(f"cholesky {dtype.__name__} n={n} kd={kd}", flush=True)
        rng = np.random.default_rng(n + kd)
        A = rng.uniform(-1, 1, (kd + 1, n))
        A[kd] = kd + 2 + rng.random(n)
        A[0, n // 2] = -0.0
        for c in range(kd):
            A[: kd - c, c] = np.nan
        ab = np.asfortranarray(A.astype(dtype))

        def run():
            x, info = bh.DeviceArray.from_numpy(ab), C.c_int64(-7)
            bh._lib.call(f"bh_{FP[dtype]}pbtrf", b"U", n, kd, x.ptr, kd + 1, C.byref(info))
            return x.numpy(), info.value

        on, off = _both(monkeypatch, run)
        assert off[1] == 0
        _same(on, off)


def test_other_stream_captured(bh, monkeypatch):
    """A call that waits for nothing, of a new thread, whose buffers are allocated by it, while another stream is
    captured: that stays valid.  (Calls that read a result back, like pbtrf, are refused then, cut or not.)"""
    hip = C.CDLL(bh._lib.LIB_PATH)  # the runtime's own symbols, through the library's dependency on it
    n, k = 300007, 3
    ab = np.ones((k + 1, n), order="F")
    ab[k] = 9
    A, b = bh.DeviceArray.from_numpy(ab), np.random.default_rng(3).standard_normal(n)

    def solve(x, errors):
        try:
            bh._lib.call("bh_dtbsv", b"U", b"N", b"N", n, k, A.ptr, k + 1, x.ptr, 1)
        except Exception as e:
            errors.append(e)

    def run():
        x, errors = bh.DeviceArray.from_numpy(b), []
        a, g = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamCreate(C.byref(a)) == 0
        assert hip.hipStreamBeginCapture(a, C.c_int(0)) == 0
        t = threading.Thread(target=solve, args=(x, errors))
        t.start()
        t.join()
        assert hip.hipStreamEndCapture(a, C.byref(g)) == 0
        if g.value:
            assert hip.hipGraphDestroy(g) == 0
        assert hip.hipStreamDestroy(a) == 0
        assert not errors
        return (x.numpy(),)

    x = bh.DeviceArray.from_numpy(b)
    solve(x, [])  # the kernels loaded before the capture
    _same(*_both(monkeypatch, run))


def test_stream_destroyed_and_another_created(bh, monkeypatch):
    """Solves on streams that are destroyed right after them, before their work has ended; a new stream may have
    the old one's handle, and its solve takes the same buffer: behind that work all the same."""
    monkeypatch.delenv("BANDEDHIP_CUT", raising=False)
    hip = C.CDLL(bh._lib.LIB_PATH)
    n, k = 400003, 5
    rng = np.random.default_rng(5)
    A = bh.DeviceArray.from_numpy(_triangle(rng, n, k, True, np.float64, "dominant"))
    b = [rng.standard_normal(n) for _ in range(6)]

    def solve(x):
        bh._lib.call("bh_dtbsv", b"U", b"N", b"N", n, k, A.ptr, k + 1, x.ptr, 1)

    want = [bh.DeviceArray.from_numpy(v) for v in b]
    for x in want:
        solve(x)
        bh.sync()
    got = [bh.DeviceArray.from_numpy(v) for v in b]
    try:
        for x in got:
            s = C.c_void_p()
            assert hip.hipStreamCreateWithFlags(C.byref(s), C.c_uint(1)) == 0
            bh._lib.call("bh_set_stream", s)
            solve(x)
            bh._lib.call("bh_set_stream", None)
            assert hip.hipStreamDestroy(s) == 0
    finally:
        bh._lib.call("bh_set_stream", None)
    assert hip.hipDeviceSynchronize() == 0
    for g, w in zip(got, want):
        _same((g.numpy(),), (w.numpy(),))


def test_kept_buffer_used_while_another_stream_is_captured(bh, monkeypatch):
    """The second and third call of a thread take its buffer again, while another stream is captured in the global
    mode: that capture stays valid, and the results are those outside of it."""
    monkeypatch.delenv("BANDEDHIP_CUT", raising=False)
    hip = C.CDLL(bh._lib.LIB_PATH)
    n, k = 30011, 3
    ab = np.ones((k + 1, n), order="F")
    ab[k] = 9
    A, b = bh.DeviceArray.from_numpy(ab), np.random.default_rng(4).standard_normal(n)
    xs = [bh.DeviceArray.from_numpy(b) for _ in range(4)]
    errors = []

    def solve(x):
        try:
            bh._lib.call("bh_dtbsv", b"U", b"N", b"N", n, k, A.ptr, k + 1, x.ptr, 1)
        except Exception as e:
            errors.append(e)

    solve(xs[0])
    bh.sync()
    a, g = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(a)) == 0
    assert hip.hipStreamBeginCapture(a, C.c_int(0)) == 0
    t = threading.Thread(target=lambda: [solve(x) for x in xs[1:]])
    t.start()
    t.join()
    assert hip.hipStreamEndCapture(a, C.byref(g)) == 0
    if g.value:
        assert hip.hipGraphDestroy(g) == 0
    assert hip.hipStreamDestroy(a) == 0
    assert not errors
    want = xs[0].numpy()
    for x in xs[1:]:
        _same((x.numpy(),), (want,))
