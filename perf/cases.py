"""The work this library is measured on: its public operations over the sizes they are used at.

Each case is a plain dict: `op` names the operation, the rest are its sizes and options.  `listed()`
gives the fixed cases, `draw(rng)` further ones of the same ranges; `prepare` makes the inputs and the
plans a program keeps, `run` is one pass through the public entry points, `work` is what the operation
cannot do without, and `exact` is its result in 64 bits from numpy alone.

Band arrays are held here as torch tensors of shape (columns, bands), which is the column-major
(bands x columns) storage of the library: entry (i, j) of a matrix with bandwidths (l, u) is at
[j, u + i - j].
"""
from __future__ import annotations

import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bandedmatrices.jl_amd"))

import banded_hip as bh  # noqa: E402
from banded_hip import _lib  # noqa: E402

BATCH_CLASSES = ((1, 1), (2, 2), (4, 3), (8, 8))


# ------------------------------------------------------------------ cases
def listed():
    return [
        # a tridiagonal-sized operator applied once per step of a time integrator: the smallest call
        {"name": "mul_small", "op": "mul", "m": 10000, "n": 10000, "l": 4, "u": 3, "dtype": "f64", "trans": "N",
         "nrhs": 0, "beta": 0.0},
        # the same product of a long discretised operator, one vector
        {"name": "mul_large", "op": "mul", "m": 1 << 20, "n": 1 << 20, "l": 8, "u": 8, "dtype": "f64", "trans": "N",
         "nrhs": 0, "beta": 0.0},
        # A'x of a rectangular operator of odd sizes in single precision (a gradient's or a Krylov method's adjoint)
        {"name": "mul_adjoint_f32", "op": "mul", "m": 1000003, "n": 999999, "l": 7, "u": 9, "dtype": "f32",
         "trans": "T", "nrhs": 0, "beta": 0.0},
        # one operator applied to a block of 64 vectors
        {"name": "mul_64_vectors", "op": "mul", "m": 1 << 20, "n": 1 << 20, "l": 8, "u": 8, "dtype": "f64",
         "trans": "N", "nrhs": 64, "beta": 0.0},
        # operators composed: banded times banded
        {"name": "matmul_banded", "op": "matmul", "n": 1 << 20, "l": 8, "u": 8, "bl": 4, "bu": 4, "dtype": "f64"},
        # A \ b of one narrow system whose rows are interchanged (a random band, no dominant diagonal; as many bands
        # below as above, since others are too ill-conditioned at this length to have a solution worth the name)
        {"name": "solve_narrow", "op": "solve", "n": 10000, "l": 4, "u": 4, "dtype": "f64", "dominant": False},
        # A \ B of a wide band with 16 right-hand sides, single-precision factors refined to double
        {"name": "solve_mixed_wide", "op": "mixed", "n": 65536, "l": 128, "u": 128, "nrhs": 16},
        # reverse-mode gradient of a loss over A \ b and A x
        {"name": "gradient", "op": "gradient", "n": 262144, "l": 16, "u": 16},
        # thousands of independent systems of mixed sizes, factored and solved
        {"name": "batch_solve", "op": "batch", "nsys": 4096, "nmax": 8192, "dtype": "f64"},
        # a QR solve of a long narrow random band
        {"name": "qr_solve", "op": "qr", "m": 100000, "n": 100000, "l": 4, "u": 4, "dtype": "f64", "dominant": False},
        # a symmetric positive definite band: factor and solve
        {"name": "cholesky_solve", "op": "cholesky", "n": 65536, "k": 8, "uplo": "U", "dtype": "f64"},
        # a triangular band solve, as a preconditioner applies it
        {"name": "triangular_solve", "op": "triangular", "n": 1 << 20, "k": 8, "uplo": "U", "trans": "N",
         "dtype": "f64"},
    ]


def _size(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["mul", "mul", "mul", "matmul", "solve", "mixed", "gradient", "batch", "qr", "cholesky",
                     "triangular"])
    dtype = rng.choice(["f64", "f64", "f32"])
    if op == "mul":
        nrhs = rng.choice([0, 0, 0, rng.randint(1, 16), rng.randint(17, 64)])
        n = _size(rng, 1000, 1 << 20)
        return {"op": op, "m": n + rng.randint(-2, 2), "n": n, "l": rng.randint(0, 8), "u": rng.randint(0, 8),
                "dtype": dtype, "trans": rng.choice(["N", "N", "T"]), "nrhs": nrhs, "beta": rng.choice([0.0, 0.0, 0.5])}
    if op == "matmul":
        return {"op": op, "n": _size(rng, 1000, 1 << 20), "l": rng.randint(0, 8), "u": rng.randint(0, 8),
                "bl": rng.randint(0, 4), "bu": rng.randint(0, 4), "dtype": dtype}
    if op == "solve":
        # single precision only where the condition number leaves it digits
        dominant, l = dtype == "f32" or rng.random() < 0.5, rng.randint(1, 8)
        return {"op": op, "n": _size(rng, 1000, 65536), "l": l, "u": rng.randint(1, 8) if dominant else l,
                "dtype": dtype, "dominant": dominant}
    if op == "mixed":
        return {"op": op, "n": _size(rng, 4096, 65536), "l": rng.randint(32, 128), "u": rng.randint(32, 128),
                "nrhs": rng.randint(1, 16)}
    if op == "gradient":
        return {"op": op, "n": _size(rng, 4096, 262144), "l": rng.randint(2, 16), "u": rng.randint(2, 16)}
    if op == "batch":
        return {"op": op, "nsys": _size(rng, 64, 4096), "nmax": _size(rng, 512, 8192), "dtype": dtype}
    if op == "qr":
        n, dominant, l = _size(rng, 1000, 100000), rng.random() < 0.5, rng.randint(1, 4)
        return {"op": op, "m": n + rng.choice([0, 0, l]), "n": n, "l": l, "u": rng.randint(1, 4) if dominant else l,
                "dtype": "f64", "dominant": dominant}
    if op == "cholesky":
        return {"op": op, "n": _size(rng, 1000, 65536), "k": rng.randint(2, 16), "uplo": rng.choice(["U", "L"]),
                "dtype": dtype}
    return {"op": op, "n": _size(rng, 1000, 1 << 20), "k": rng.randint(2, 16), "uplo": rng.choice(["U", "L"]),
            "trans": rng.choice(["N", "T"]), "dtype": dtype}


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.float64


def _lu_flops(n, l, u):
    return n * (l + 2 * l * (l + u))


def _batch_sizes(case):
    """(n, kl, ku) of every system: n log-uniform in [256, nmax] (64 .. for short batches), classes in turn."""
    nsys, nmax = case["nsys"], case["nmax"]
    nmin = min(256, nmax // 2)
    n = [int(round(nmin * (nmax / nmin) ** ((s + 0.5) / nsys))) for s in range(nsys)]
    random.Random(nsys * 10007 + nmax).shuffle(n)
    kl = [BATCH_CLASSES[s % 4][0] for s in range(nsys)]
    ku = [BATCH_CLASSES[s % 4][1] for s in range(nsys)]
    return n, kl, ku


def work(case):
    op, w = case["op"], 4 if case.get("dtype") == "f32" else 8
    n = case.get("n", 0)
    if op == "mul":
        h, r = case["l"] + case["u"] + 1, max(1, case["nrhs"])
        out = case["m"] if case["trans"] == "N" else n
        return {"bytes": w * (h * n + r * (n + case["m"]) + (r * out if case["beta"] else 0)), "flops": 2 * h * n * r}
    if op == "matmul":
        ha, hb = case["l"] + case["u"] + 1, case["bl"] + case["bu"] + 1
        return {"bytes": w * n * (ha + hb + ha + hb - 1), "flops": 2 * ha * hb * n}
    l, u = case.get("l", 0), case.get("u", 0)
    if op == "solve":
        return {"bytes": w * n * (l + u + 3), "flops": _lu_flops(n, l, u) + 2 * n * (2 * l + u)}
    if op == "mixed":
        r = case["nrhs"]
        return {"bytes": 8 * n * (l + u + 1 + 2 * r), "flops": _lu_flops(n, l, u) + 2 * n * r * (2 * l + u)}
    if op == "gradient":
        return {"bytes": 8 * n * (2 * (l + u + 1) + 5), "flops": _lu_flops(n, l, u) + 4 * n * (2 * l + u) + 5 * n * (l + u + 1)}
    if op == "batch":
        rows = list(zip(*_batch_sizes(case)))
        return {"bytes": sum(k * (w * (2 * (2 * p + q + 1) + 2) + 8) for k, p, q in rows),
                "flops": sum(_lu_flops(k, p, q) + 2 * k * (2 * p + q) for k, p, q in rows)}
    if op == "qr":
        return {"bytes": w * (n * (l + u + 1) + case["m"] + n), "flops": n * (4 * (l + 1) * (l + u) + 4 * (l + 1) + 2 * (l + u))}
    k = case["k"]
    if op == "cholesky":
        return {"bytes": w * n * (k + 3), "flops": n * (k * (k + 3) + 4 * k)}
    return {"bytes": w * n * (k + 3), "flops": 2 * n * k}


# ------------------------------------------------------------------ inputs
def _inputs(case, seed):
    """The tensors of one problem, on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, op, n = _dtype(case), case["op"], case.get("n", 0)

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device="cuda", dtype=dt)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dt)

    if op == "mul":
        rows, cols = (case["m"], n) if case["trans"] == "N" else (n, case["m"])
        r = case["nrhs"]
        return {"A": normal(n, case["l"] + case["u"] + 1), "x": normal(*((r, cols) if r else (cols,))),
                "y": normal(*((r, rows) if r else (rows,)))}
    if op == "matmul":
        return {"A": normal(n, case["l"] + case["u"] + 1), "B": normal(n, case["bl"] + case["bu"] + 1)}
    if op in ("solve", "qr"):
        A = uniform(n, case["l"] + case["u"] + 1)
        if case["dominant"]:
            A[:, case["u"]] += case["l"] + case["u"] + 1
        return {"A": A, "b": normal(case.get("m", n))}
    if op == "mixed":
        A = normal(n, case["l"] + case["u"] + 1)
        A[:, case["u"]] += 2 * (case["l"] + case["u"])
        return {"A": A, "B": normal(case["nrhs"], n)}
    if op == "gradient":
        A = normal(n, case["l"] + case["u"] + 1)
        A[:, case["u"]] += 2 * (case["l"] + case["u"])
        return {"A": A, "b": normal(n), "w": normal(n), "x0": normal(n)}
    if op == "batch":
        sizes, kl, ku = _batch_sizes(case)
        bands, b = [], normal(sum(sizes))
        for k, p, q in zip(sizes, kl, ku):
            A = uniform(k, p + q + 1)
            A[:, q] += p + q + 1
            bands.append(A)
        return {"bands": bands, "b": b}
    k = case["k"]
    A = uniform(n, k + 1) * 2 - 1
    diagonal = k if case["uplo"] == "U" else 0
    if op == "cholesky":
        A[:, diagonal] = k + 1 + uniform(n)
    else:
        A *= 0.5 / k
        A[:, diagonal] = 1 + uniform(n)
    return {"A": A, "b": normal(n)}


class _Memory:
    """A DeviceArray's memory as torch.as_tensor takes it; keeps the array alive."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": tuple(reversed(array.shape)), "typestr": array.dtype.str,
                                         "data": (array.ptr, False), "strides": None, "version": 2}


def _tensor(array):
    return torch.as_tensor(_Memory(array), device="cuda")


def _array(t):
    """A DeviceArray holding a copy of the tensor (its axes reversed: column-major)."""
    d = bh.DeviceArray(tuple(reversed(t.shape)), np.float32 if t.dtype == torch.float32 else np.float64)
    _tensor(d).copy_(t)
    return d


def _matrix(t, m, l, u):
    return bh.BandedMatrix(_array(t), m, l, u)


def _triangle(case, A):
    k = case["k"]
    return _matrix(A, case["n"], *((0, k) if case["uplo"] == "U" else (k, 0)))


def prepare(case, seed):
    op, n, t = case["op"], case.get("n", 0), _inputs(case, seed)
    s = {"case": case}
    if op == "mul":
        s["A"], s["x"], s["y"] = _matrix(t["A"], case["m"], case["l"], case["u"]), _array(t["x"]), _array(t["y"])
        s["out"] = _tensor(s["y"])
    elif op == "matmul":
        s["A"] = _matrix(t["A"], n, case["l"], case["u"])
        s["B"] = _matrix(t["B"], n, case["bl"], case["bu"])
        s["C"] = bh.BandedMatrix.zeros((n, n), (case["l"] + case["bl"], case["u"] + case["bu"]), s["A"].dtype)
        s["out"] = _tensor(s["C"].data)
    elif op == "mixed":
        s["A"], s["B"] = _matrix(t["A"], n, case["l"], case["u"]), _array(t["B"])
        s["X"] = bh.DeviceArray((n, case["nrhs"]))
        s["solver"] = bh.MixedSolver(n, case["l"], case["u"], case["nrhs"])
        s["out"] = _tensor(s["X"])
    elif op == "gradient":
        s["A"] = _matrix(t["A"], n, case["l"], case["u"])
        s["b"], s["w"], s["x0"] = _array(t["b"]), _array(t["w"]), _array(t["x0"])
    elif op == "batch":
        sizes, kl, ku = _batch_sizes(case)
        plan = bh.BatchedGBSV(sizes, kl, ku, np.float32 if case["dtype"] == "f32" else np.float64)
        s["plan"] = plan
        s["AB"], s["B"] = bh.DeviceArray.zeros(plan.AB.shape, plan.dtype), _array(t["b"])
        bh.sync()
        AB = _tensor(s["AB"])
        for k, (A, p, q) in enumerate(zip(t["bands"], kl, ku)):
            ld, at = 2 * p + q + 1, int(plan.ab_off[k])
            AB[at:at + ld * sizes[k]].view(sizes[k], ld)[:, p:] = A
        s["out"] = {"x": _tensor(plan.B), "factors": _tensor(plan.AB), "ipiv": _tensor(plan.ipiv),
                    "info": _tensor(plan.info)}
    elif op in ("solve", "qr"):
        s["A"], s["b"] = _matrix(t["A"], case.get("m", n), case["l"], case["u"]), _array(t["b"])
    else:
        s["A"], s["b"] = _triangle(case, t["A"]), _array(t["b"])
        if op == "triangular":
            s["T"] = (bh.UpperTriangular if case["uplo"] == "U" else bh.LowerTriangular)(s["A"])
    torch.cuda.synchronize()
    bh.sync()
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    op = case["op"]
    if op == "mul":
        bh.mul(s["y"], s["A"], s["x"], 1.0, case["beta"], case["trans"])
        return s["out"]
    if op == "matmul":
        bh.gbmm(s["A"], s["B"], s["C"])
        return s["out"]
    if op == "solve":
        return _tensor(bh.solve(s["A"], s["b"]))
    if op == "mixed":
        s["solver"].solve(s["A"], s["B"], s["X"])
        return s["out"]
    if op == "gradient":
        loss, dA, db, x = bh.loss_and_grad(s["A"], s["b"], s["w"], s["x0"])
        return {"loss": loss, "dA": _tensor(dA.data), "db": _tensor(db), "x": _tensor(x)}
    if op == "batch":
        # the solve is in place: a program that steps in time writes its matrices and right-hand sides anew
        plan = s["plan"]
        _lib.call("bh_memcpy_dtod", plan.AB.ptr, s["AB"].ptr, plan.AB.nbytes)
        _lib.call("bh_memcpy_dtod", plan.B.ptr, s["B"].ptr, plan.B.nbytes)
        plan.solve()
        return s["out"]
    if op == "qr":
        return _tensor(bh.qr_solve(s["A"], s["b"]))
    if op == "cholesky":
        F = bh.cholesky(bh.Symmetric(s["A"], case["uplo"]))
        x = bh.ldiv_(F, s["b"].copy())
        return {"x": _tensor(x), "factor": _tensor(F.factors.data)}
    return _tensor(s["T"].ldiv_(s["b"].copy(), case["trans"]))


# ------------------------------------------------------------------ 64-bit results
def _transposed(A, m, l, u):
    """Band array of A' (m columns) from that of A (n columns, bandwidths l, u)."""
    n = A.shape[0]
    T = np.zeros((m, l + u + 1))
    for r in range(l + u + 1):  # entry (i, j), i = j + r - u, is entry (j, i) of A': row l + j - i = l + u - r
        j0, j1 = max(0, u - r), min(n, m + u - r)
        if j1 > j0:
            T[j0 + r - u:j1 + r - u, l + u - r] = A[j0:j1, r]
    return T


def _product(A, m, l, u, x):
    """A x; x has shape (vectors, n)."""
    n = A.shape[0]
    y = np.zeros((x.shape[0], m))
    for r in range(l + u + 1):
        j0, j1 = max(0, u - r), min(n, m + u - r)
        if j1 > j0:
            y[:, j0 + r - u:j1 + r - u] += A[j0:j1, r] * x[:, j0:j1]
    return y


def _block(A, m, l, u, i0, i1, j0, j1):
    """Rows i0..i1, columns j0..j1 of the matrix, dense."""
    n = A.shape[0]
    D = np.zeros((i1 - i0, j1 - j0))
    j1 = min(j1, n)
    i, j = np.meshgrid(np.arange(i0, min(i1, m)), np.arange(j0, j1), indexing="ij")
    r = u + i - j
    ok = (r >= 0) & (r <= l + u)
    D[i[ok] - i0, j[ok] - j0] = A[j[ok], r[ok]]
    return D


def _solved(A, m, l, u, B):
    """Least-squares solution (m >= n) of A x = b for each row of B, by Householder QR a block of columns at a
    time: the rows that a block's columns reach are reduced to R, the rest is carried to the next block."""
    n, r = A.shape[0], B.shape[0]
    if l > 0 and u == 0 and m == n:  # lower triangular: turned about, it is upper
        return _solved(np.ascontiguousarray(A[::-1, ::-1]), n, 0, l, B[:, ::-1])[:, ::-1]
    c = max(64, l + u)
    wide = c + l + u
    carry, kept, top = np.zeros((0, wide + r)), [], 0
    for j0 in range(0, n, c):
        j1 = min(n, j0 + c)
        end = m if j1 == n else min(m, j1 + l)
        new = np.hstack([_block(A, m, l, u, top, end, j0, j0 + wide), B[:, top:end].T])
        top, both = end, np.vstack([carry, new])
        if l == 0:
            R = both
        else:
            R = np.linalg.qr(both, mode="r")
        kept.append(R[:j1 - j0])
        carry = np.hstack([R[j1 - j0:, c:wide], np.zeros((max(0, R.shape[0] - (j1 - j0)), c)), R[j1 - j0:, wide:]])
    x = np.zeros((n + wide, r))
    for b in range(len(kept) - 1, -1, -1):
        j0, R = b * c, kept[b]
        k = R.shape[0]
        x[j0:j0 + k] = np.linalg.solve(R[:, :k], R[:, wide:] - R[:, k:wide] @ x[j0 + k:j0 + wide])
    return np.ascontiguousarray(x[:n].T)


def _batch_solved(sizes, kl, ku, bands, b):
    """x of every system, by elimination down the columns without interchanges (the diagonals dominate), over
    all systems of one class at once."""
    at = np.concatenate([[0], np.cumsum(sizes)])
    x = torch.zeros_like(b)
    for p, q in BATCH_CLASSES:
        group = [s for s in range(len(sizes)) if (kl[s], ku[s]) == (p, q)]
        if not group:
            continue
        longest = max(sizes[s] for s in group)
        # rows[i, s, :]: row i of system s, columns i - p .. i + q; rows past a system's end are the identity's
        rows = torch.zeros(longest + p, len(group), p + q + 1, dtype=torch.float64, device=b.device)
        rows[:, :, p] = 1
        f = torch.zeros(longest + q, len(group), dtype=torch.float64, device=b.device)
        for g, s in enumerate(group):
            k, A = sizes[s], bands[s].double()
            for r in range(p + q + 1):
                j0, j1 = max(0, q - r), min(k, k + q - r)
                rows[j0 + r - q:j1 + r - q, g, p + q - r] = A[j0:j1, r]
            f[:k, g] = b[at[s]:at[s] + k]
        for j in range(longest):
            for i in range(1, p + 1):
                lead = p - i  # column j in row j + i
                t = rows[j + i, :, lead] / rows[j, :, p]
                rows[j + i, :, lead + 1:lead + 1 + q] -= t[:, None] * rows[j, :, p + 1:]
                if j + i < longest:
                    f[j + i] -= t * f[j]
        for j in range(longest - 1, -1, -1):
            f[j] = (f[j] - (rows[j, :, p + 1:] * f[j + 1:j + 1 + q].T).sum(1)) / rows[j, :, p]
        for g, s in enumerate(group):
            x[at[s]:at[s] + sizes[s]] = f[:sizes[s], g]
    return x


def exact(case, seed):
    op, n, t = case["op"], case.get("n", 0), _inputs(case, seed)
    l, u = case.get("l", 0), case.get("u", 0)
    if op == "batch":
        sizes, kl, ku = _batch_sizes(case)
        return {"x": _batch_solved(sizes, kl, ku, t["bands"], t["b"].double()), "factors": None, "ipiv": None,
                "info": None}
    h = {k: v.double().cpu().numpy() for k, v in t.items()}
    A = h["A"]
    if op == "mul":
        x, y = np.atleast_2d(h["x"]), np.atleast_2d(h["y"])
        if case["trans"] == "N":
            z = _product(A, case["m"], l, u, x)
        else:
            z = _product(_transposed(A, case["m"], l, u), n, u, l, x)
        z = z + case["beta"] * y
        return z if case["nrhs"] else z[0]
    if op == "matmul":
        B, ha, bu = h["B"], l + u + 1, case["bu"]
        C, j = np.zeros((n, ha + B.shape[1] - 1)), np.arange(n)
        for r in range(ha):  # zero the slots of A outside the matrix
            k = j + r - u
            A[(k < 0) | (k >= n), r] = 0
        for r in range(B.shape[1]):
            k = j + r - bu
            ok = (k >= 0) & (k < n)
            C[ok, r:r + ha] += A[k[ok]] * B[ok, r][:, None]
        return C
    if op == "solve":
        return _solved(A, n, l, u, h["b"][None])[0]
    if op == "mixed":
        return _solved(A, n, l, u, h["B"])
    if op == "gradient":
        x = _solved(A, n, l, u, h["b"][None])[0]
        lam = _solved(_transposed(A, n, l, u), n, u, l, h["w"][None])[0]
        y = _product(A, n, l, u, h["x0"][None])[0]
        dA = np.zeros_like(A)
        for r in range(l + u + 1):
            j0, j1 = max(0, u - r), min(n, n + u - r)
            i = slice(j0 + r - u, j1 + r - u)
            dA[j0:j1, r] = y[i] * h["x0"][j0:j1] - lam[i] * x[j0:j1]
        return {"loss": float(h["w"] @ x + 0.5 * (y @ y)), "dA": dA, "db": lam, "x": x}
    if op == "qr":
        x = _solved(A, case["m"], l, u, h["b"][None])[0]
        if case["m"] == n:
            return x
        return None  # the rows past the solution hold the residual's coordinates
    k = case["k"]
    l, u = (0, k) if case["uplo"] == "U" else (k, 0)
    if op == "cholesky":
        upper, lower = A, _transposed(A, n, l, u)
        if case["uplo"] == "L":
            upper, lower = lower, upper
        full = np.zeros((n, 2 * k + 1))
        full[:, k:] = lower
        full[:, :k + 1] = upper
        for r in range(k):  # slots outside the matrix
            full[:k - r, r] = 0
            full[n - k + r:, 2 * k - r] = 0
        return {"x": _solved(full, n, k, k, h["b"][None])[0], "factor": None}
    if case["trans"] == "T":
        A, l, u = _transposed(A, n, l, u), u, l
    return _solved(A, n, l, u, h["b"][None])[0]
