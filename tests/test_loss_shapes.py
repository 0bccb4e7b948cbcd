"""CPU: loss_and_grad refuses right-hand sides and weights that are not one
vector before any work, instead of returning the loss of their first column
(the device sums take bare pointers).  GPU: what it accepts, and the loss
itself in both precisions against a 64-bit sum on the host."""
import numpy as np
import pytest

import banded_hip
from banded_hip import adjoint
from banded_hip.bandedmatrix import DimensionMismatch

from _util import band


class _Shaped:
    """Stands for a device array or matrix whose shape is all that is looked at."""

    dtype = np.dtype(np.float64)

    def __init__(self, *shape):
        self.shape = shape


@pytest.mark.parametrize("b,w", [((8, 2), (8,)), ((8, 8), (8,)), ((8,), (8, 1)), ((8,), (8, 3)), ((8, 2), (8, 2)), ((7,), (8,)),
                                 ((8,), (9,)), ((8, 0), (8,)), ((1, 8), (8,))])
def test_refused_before_any_work(monkeypatch, b, w):
    def reached(*a, **k):
        raise AssertionError("work began")

    monkeypatch.setattr(adjoint, "lu", reached)
    with pytest.raises(DimensionMismatch):
        banded_hip.loss_and_grad(_Shaped(8, 8), _Shaped(*b), _Shaped(*w), _Shaped(8))


@pytest.mark.gpu
def test_several_columns_refused_on_the_device(bh):
    n = 50
    rng = np.random.default_rng(0)
    A = band(rng, 2, 1, n)
    A[1] += 8
    dev = lambda *shape: bh.DeviceArray.from_numpy(np.asfortranarray(rng.standard_normal(shape)))
    M = bh.BandedMatrix.from_host(A, n, 2, 1)
    with pytest.raises(ValueError):
        bh.loss_and_grad(M, dev(n, 2), dev(n), dev(n))
    with pytest.raises(ValueError):
        bh.loss_and_grad(M, dev(n), dev(n, 1), dev(n))
    b, w, x0 = dev(n), dev(n), dev(n)
    one = bh.DeviceArray.from_numpy(b.numpy().reshape(n, 1))
    L, dA, db, x = bh.loss_and_grad(M, b, w, x0)
    L1, dA1, db1, x1 = bh.loss_and_grad(M, one, w, x0)
    assert L1 == L and x1.shape == (n, 1) and np.array_equal(x1.numpy()[:, 0], x.numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [0, 1, 63, 256, 257, 65535, 65537, 200001])
def test_loss_sum(bh, dtype, n):
    """Products and sums are in double for both types: a thread adds its n / 65536 terms, then some 20 sums across
    threads and workgroups, each rounded once."""
    import ctypes as C

    rng = np.random.default_rng(n)
    w, x, y = (rng.standard_normal(n).astype(dtype) for _ in range(3))
    d = [bh.DeviceArray.from_numpy(v) for v in (w, x, y)]
    L = C.c_double(-1.0)
    bh._lib.call(f"bh_{'d' if dtype == np.float64 else 's'}gb_loss", n, *[v.ptr for v in d], C.byref(L))
    w, x, y = (v.astype(np.longdouble) for v in (w, x, y))
    terms = w * x + y * y / 2
    size = float(np.sum(np.abs(w * x)) + np.sum(y * y / 2))
    assert abs(L.value - float(np.sum(terms))) <= (4 + 2 * (n // 65536 + 20)) * 2.0 ** -53 * size
