"""CPU: the bookkeeping of the blocks that bh_free keeps (csrc/bh_blocks.hpp),
compiled for the host against a device that only counts.  GPU: a block freed
twice is an error through the C ABI, and the blocks handed out stay distinct."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HOST = r"""
#include <stdio.h>
#include <stdlib.h>
#include <set>
#include "bh_blocks.hpp"
// Addresses are numbers: alloc hands out new ones, release of one that is not
// live is what a runtime reports (and what must never be asked for a kept block).
struct State { std::set<void*> live; size_t next = 4096, limit = ~size_t(0), bytes = 0; int released = 0, bad = 0, fail_wait = 0;
               size_t elsewhere = 0;
               std::set<size_t> sizes; size_t size_of[4096]; };
static State S;
struct Dev {
    static constexpr int kNoMemory = 2, kBadPointer = 1;
    int current(int *d) { *d = 0; return 0; }
    int alloc(void **p, size_t n) {
        if (S.bytes + n > S.limit) return kNoMemory;
        *p = (void*)S.next; S.next += 4096; S.live.insert(*p); S.size_of[(size_t)*p / 4096] = n; S.bytes += n; return 0;
    }
    int release(void *p) {
        if (!S.live.erase(p)) { ++S.bad; return kBadPointer; }
        S.bytes -= S.size_of[(size_t)p / 4096]; ++S.released; return 0;
    }
    int wait() { return S.fail_wait; }
    void others() { S.bytes -= S.elsewhere; S.elsewhere = 0; }
};
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
typedef bh::BlockCache<Dev> Cache;
static const size_t M = size_t(1) << 20;
CASES
"""

CASES = {
    "twice": r"""
int main() {  // the second free of a kept block is an error, and the block stays whole for the next take
    Cache c; void *p, *q, *r;
    CHECK(c.take(&p, 16 * M) == 0 && c.give(p) == 0 && c.kept_bytes() == 16 * M);
    CHECK(c.give(p) == Dev::kBadPointer && S.live.count(p) == 1 && c.kept_bytes() == 16 * M);
    CHECK(c.take(&q, 16 * M) == 0 && q == p && S.live.count(q) == 1);
    CHECK(c.take(&r, 16 * M) == 0 && r != q);
    CHECK(c.give(q) == 0 && c.give(r) == 0 && c.give(q) != 0 && c.give(r) != 0 && S.bad == 0);
    return 0;
}""",
    "small": r"""
int main() {  // small and very large blocks go back at once; freeing them again is the runtime's error
    Cache c; void *p;
    CHECK(c.take(&p, M) == 0 && c.give(p) == 0 && c.kept_bytes() == 0 && S.live.empty());
    CHECK(c.give(p) == Dev::kBadPointer);
    CHECK(c.take(&p, 600 * M) == 0 && c.give(p) == 0 && c.kept_bytes() == 0 && S.live.empty());
    CHECK(c.give(p) == Dev::kBadPointer);
    return 0;
}""",
    "bounded": r"""
int main() {  // never more than kKeep kept, the oldest go first, and unused ones after kAge frees
    Cache c; void *p[40];
    for (int i = 0; i < 40; ++i) CHECK(c.take(&p[i], 100 * M) == 0);
    for (int i = 0; i < 40; ++i) CHECK(c.give(p[i]) == 0 && c.kept_bytes() <= Cache::kKeep);
    CHECK(c.kept_bytes() == 1000 * M && S.live.size() == 10 && S.live.count(p[39]) && !S.live.count(p[0]));
    void *q;
    for (int i = 0; i < 80; ++i) CHECK(c.take(&q, 10 * M) == 0 && c.give(q) == 0);
    CHECK(c.kept_bytes() == 10 * M && S.live.size() == 1 && S.bad == 0);
    return 0;
}""",
    "wait_fails": r"""
int main() {  // a free whose wait fails has freed nothing: the block is in use still, and a second try frees it
    Cache c; void *p, *q;
    CHECK(c.take(&p, 16 * M) == 0);
    S.fail_wait = 7;
    CHECK(c.give(p) == 7 && S.live.count(p) == 1 && c.kept_bytes() == 0);
    CHECK(c.take(&q, 16 * M) == 0 && q != p);
    S.fail_wait = 0;
    CHECK(c.give(p) == 0 && c.give(p) == Dev::kBadPointer && c.give(q) == 0 && S.bad == 0 && c.kept_bytes() == 32 * M);
    return 0;
}""",
    "out_of_memory": r"""
int main() {  // a request of any size has the kept blocks, and what is kept elsewhere, given back before it fails
    for (size_t want : {size_t(4096), M, 16 * M, 64 * M}) {
        Cache c; void *p, *q;
        S = State(); S.limit = 100 * M;
        CHECK(c.take(&p, 48 * M) == 0 && c.take(&q, 48 * M) == 0 && c.give(p) == 0 && c.give(q) == 0);
        S.limit = 96 * M;
        CHECK(c.take(&p, want) == 0 && c.kept_bytes() == 0 && S.bytes == want);
        S.elsewhere = S.limit - S.bytes; S.bytes = S.limit;
        CHECK(c.take(&q, want / 4) == 0 && S.elsewhere == 0);
        CHECK(c.take(&q, 97 * M) == Dev::kNoMemory && S.bad == 0);
    }
    Cache c; void *p;
    S = State();
    CHECK(c.take(&p, 48 * M) == 0 && c.give(p) == 0);
    c.drop();
    CHECK(c.kept_bytes() == 0 && S.live.empty() && c.give(p) == Dev::kBadPointer);
    return 0;
}""",
}


def _run(tmp_path, name):
    src = tmp_path / f"{name}.cpp"
    src.write_text(HOST.replace("CASES", CASES[name]))
    exe = tmp_path / name
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "bandedmatrices.jl_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("name", list(CASES))
def test_bookkeeping(tmp_path, name):
    _run(tmp_path, name)


@pytest.mark.gpu
def test_freed_twice(bh):
    L, n = bh.load_library(), 24 << 20
    p, q, r = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert L.bh_malloc(C.byref(p), n) == 0 and L.bh_free(p) == 0
    assert L.bh_free(p) != 0
    assert L.bh_malloc(C.byref(q), n) == 0 and L.bh_malloc(C.byref(r), n) == 0 and q.value != r.value
    a, b = np.full(n, 3, np.uint8), np.full(n, 5, np.uint8)
    for v, h in ((q, a), (r, b)):
        assert L.bh_memcpy_htod(v, h.ctypes.data, n) == 0
    got = np.zeros(n, np.uint8)
    for v, h in ((q, a), (r, b)):
        assert L.bh_memcpy_dtoh(got.ctypes.data, v, n) == 0 and np.array_equal(got, h)
    assert L.bh_free(q) == 0 and L.bh_free(r) == 0 and L.bh_free(q) != 0


def _free_bytes(bh):
    hip = C.CDLL(bh._lib.LIB_PATH)  # the runtime's own symbols, through the library's dependency on it
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.gpu
def test_trim_gives_back(bh):
    """What the library keeps goes back on request: freed blocks, and the block paths' buffers of every thread,
    one that lives on included; later calls work as before."""
    import gc
    import threading

    n, kl, ku = 200000, 4, 4
    h = np.ones((2 * kl + ku + 1, n), order="F")
    h[kl + ku] = 40

    def factor():
        d, p, info = bh.DeviceArray.from_numpy(h), bh.DeviceArray((n,), np.int64), C.c_int64(-1)
        bh._lib.call("bh_dgbtrf", n, n, kl, ku, d.ptr, 2 * kl + ku + 1, p.ptr, C.byref(info))
        assert info.value == 0
        return d.numpy()

    first = factor()
    gc.collect()  # arrays that earlier tests left
    bh.trim()
    base = _free_bytes(bh)
    a = bh.DeviceArray((64 << 20,), np.uint8)
    a.free()
    assert _free_bytes(bh) <= base - (64 << 20)
    go, done, out = threading.Event(), threading.Event(), []

    def other():
        out.append(factor())
        done.set()
        go.wait(60)
        out.append(factor())

    t = threading.Thread(target=other)
    t.start()
    assert done.wait(60)
    held = base - _free_bytes(bh)
    assert held >= (64 << 20) + n * (2 * kl + ku + 1) * 8  # the block, the thread's copies of the matrix
    bh.trim()
    assert base - _free_bytes(bh) <= 8 << 20
    go.set()
    t.join(60)
    assert len(out) == 2 and all(o.tobytes() == first.tobytes() for o in out)
