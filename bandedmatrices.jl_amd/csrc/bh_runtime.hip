// bh_runtime.hip -- device selection, memory, stream and event plumbing.
#include <stdarg.h>
#include <stdio.h>

#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "bh_blocks.hpp"
#include "bh_common.hpp"
#include "bh_cut.hpp"

namespace bh {

static thread_local char g_err[512] = "";
static thread_local hipStream_t g_user_stream = nullptr;
static hipStream_t g_own_stream = nullptr;
static int g_device = -1;
// Library-owned device memory (allocated by bh_init, grown only when a call
// needs more than any earlier one): the entry points take their info words,
// flags and temporaries from here instead of allocating per call.  Calls are
// stream-ordered on the library stream; calls that overlap on different
// streams must not share the library (LAPACK-like reentrancy: one handle per
// task).
static i64 *g_ctrl = nullptr;
static void *g_scratch = nullptr;
static size_t g_scratch_bytes = 0;
constexpr size_t kCtrlBytes = 256;
constexpr size_t kScratchInitial = 8u << 20;

void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int hip_fail(hipError_t e, const char *what, const char *file, int line) {
    set_error("%s failed: %s (%s:%d)", what, hipGetErrorString(e), file, line);
    return e == hipErrorOutOfMemory ? BH_ERR_ALLOC : BH_ERR_HIP;
}

static int ensure_init() {
    if (g_device >= 0) return BH_OK;
    return bh_init(0);
}

hipStream_t stream() {
    if (g_user_stream) return g_user_stream;
    return g_own_stream;
}

int ctrl_words(i64 **p) {
    int st = ensure_init();
    if (st) return st;
    *p = g_ctrl;
    return BH_OK;
}

int scratch_buffer(size_t bytes, void **p) {
    int st = ensure_init();
    if (st) return st;
    if (bytes > g_scratch_bytes) {
        // grow: earlier work on the stream may still read the old buffer
        BH_HIP(hipStreamSynchronize(stream()));
        if (g_scratch) BH_HIP(hipFree(g_scratch));
        g_scratch = nullptr;
        g_scratch_bytes = 0;
        const size_t nb = bytes + bytes / 2;
        BH_HIP(device_alloc(&g_scratch, nb));
        g_scratch_bytes = nb;
    }
    *p = g_scratch;
    return BH_OK;
}

// ---- memory of the cut paths (bh_cut.hpp).  Each thread keeps up to four
// buffers of at most kCutKeep bytes, one to a stream, and frees them when it ends;
// a fifth stream takes over the buffer unused for longest, behind its last
// use.  (A stream-ordered pool of HIP's, tried first, cost 60-140 us a call
// with a synchronisation between calls; this costs under 5.)
struct CutBuf {
    int dev = -1;
    hipStream_t st = nullptr;
    void *p = nullptr;
    size_t bytes = 0;
    hipEvent_t done = nullptr;  // behind the last call that used it
    bool busy = false;          // a call of its thread has it: nobody else touches it
    unsigned long long used = 0;
};
// Allocations, frees and waits of a call on one stream are legal while another
// stream is captured in the global mode only from a thread whose own mode is
// relaxed; otherwise they fail and spoil that capture.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Frees a buffer behind the work that used it; false: it could not be waited for.
static bool cut_release(CutBuf &c) {
    if (!c.p) return true;
    if (hipEventSynchronize(c.done) != hipSuccess || hipFree(c.p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    c.p = nullptr;
    c.bytes = 0;
    return true;
}

struct CutBufs;
// every thread's, so that memory can be had back from all of them (never
// destroyed: threads may end after this unit's statics)
static std::mutex &g_cut_mutex = *new std::mutex;
static std::vector<CutBufs *> &g_cut_all = *new std::vector<CutBufs *>;

struct CutBufs {
    std::mutex m;  // the buffers' fields, but for those of a busy one
    CutBuf b[4];
    unsigned long long clock = 0;
    int off = 0;
    // the last call that could run by blocks: how often blocks were launched,
    // where its verdict stands (null once the buffer has gone back) or what it was
    int tries = 0, known[2] = {1, 0};
    const int *flags = nullptr;
    hipStream_t flags_st = nullptr;
    int *host = nullptr;  // pinned
    bool holds_flags(const CutBuf &c) const {
        const char *f = (const char *)flags, *p = (const char *)c.p;
        return f && p && f >= p && f < p + c.bytes;
    }
    CutBufs() {
        std::lock_guard<std::mutex> all(g_cut_mutex);
        g_cut_all.push_back(this);
    }
    ~CutBufs() {
        {
            std::lock_guard<std::mutex> all(g_cut_mutex);
            g_cut_all.erase(std::find(g_cut_all.begin(), g_cut_all.end(), this));
        }
        const RelaxedCapture relaxed;
        for (CutBuf &c : b) {
            if (c.p) (void)hipFree(c.p);
            if (c.done) (void)hipEventDestroy(c.done);
        }
        if (host) (void)hipHostFree(host);
    }
};
static thread_local CutBufs g_cut;

// The idle buffers of every thread.
static void cut_release_idle() {
    const RelaxedCapture relaxed;
    std::lock_guard<std::mutex> all(g_cut_mutex);
    for (CutBufs *t : g_cut_all) {
        std::lock_guard<std::mutex> lock(t->m);
        for (CutBuf &c : t->b) {
            if (c.busy || !c.p) continue;
            const bool noted = t->holds_flags(c);
            if (cut_release(c) && noted) {
                t->flags = nullptr;
                t->tries = 0;
            }
        }
    }
}

// ---- large blocks of bh_malloc (bh_blocks.hpp)
struct HipDevice {
    static constexpr int kNoMemory = hipErrorOutOfMemory, kBadPointer = hipErrorInvalidValue;
    int current(int *dev) { return hipGetDevice(dev); }
    int alloc(void **p, size_t bytes) {
        const hipError_t e = hipMalloc(p, bytes);
        if (e == hipErrorOutOfMemory) (void)hipGetLastError();
        return e;
    }
    int release(void *p) { return hipFree(p); }
    int wait() { return hipDeviceSynchronize(); }
    void others() { cut_release_idle(); }
};
// never destroyed: arrays may be freed while the process ends
static BlockCache<HipDevice> &g_blocks = *new BlockCache<HipDevice>;

static void release_kept() {
    g_blocks.drop();
    cut_release_idle();
}

hipError_t device_alloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    release_kept();
    return hipMalloc(p, bytes);
}

CutOff::CutOff() { ++g_cut.off; }
CutOff::~CutOff() { --g_cut.off; }

bool cut_enabled() {
    if (g_cut.off > 0) return false;
    const char *e = getenv("BANDEDHIP_CUT");
    return !(e && !strcmp(e, "off"));
}

int *cut_host_words() {
    if (!g_cut.host) {
        const RelaxedCapture relaxed;
        if (hipHostMalloc((void **)&g_cut.host, kCutWords * sizeof(int),
                          hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
            (void)hipGetLastError();
            g_cut.host = nullptr;
            return nullptr;
        }
    }
    for (int i = 0; i < kCutWords; ++i) g_cut.host[i] = -1;
    return g_cut.host;
}

int cut_poll(const int *word, hipStream_t st) {
    const RelaxedCapture relaxed;
    for (;;) {
        for (int i = 0; i < 256; ++i) {
            const int v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
            if (v >= 0) return v;
            __builtin_ia32_pause();
        }
        // (the word may come between the look at it and the stream's end)
        if (hipStreamQuery(st) != hipErrorNotReady) return __atomic_load_n(word, __ATOMIC_ACQUIRE);
    }
}

void cut_begin() {
    std::lock_guard<std::mutex> lock(g_cut.m);
    g_cut.tries = 0;
    g_cut.flags = nullptr;
}

void cut_note(const int *flags, hipStream_t st) {
    std::lock_guard<std::mutex> lock(g_cut.m);
    ++g_cut.tries;
    g_cut.flags = flags;
    g_cut.flags_st = st;
}

void *cut_alloc(size_t bytes, hipStream_t st) {
    if (bytes > kCutMax) return nullptr;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    int dev = -1;
    if (hipStreamIsCapturing(st, &cap) != hipSuccess || hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (cap != hipStreamCaptureStatusNone) return nullptr;
    CutBuf *c = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_cut.m);
        for (CutBuf &x : g_cut.b) {
            if (x.busy) continue;
            if (x.p && x.dev == dev && x.st == st) {
                c = &x;
                break;
            }
            if (!c || x.used < c->used) c = &x;
        }
        if (!c) return nullptr;
        c->busy = true;
    }
    bool ok = true;
    if (c->p && c->dev == dev && c->bytes >= bytes) {
        // also on what looks like the same stream: it may be a new one at the
        // handle of a destroyed one whose work still runs
        ok = hipStreamWaitEvent(st, c->done, 0) == hipSuccess;
    } else {
        const RelaxedCapture relaxed;
        ok = cut_release(*c);
        if (ok && c->done && c->dev != dev) {
            (void)hipEventDestroy(c->done);
            c->done = nullptr;
        }
        if (ok && !c->done) ok = hipEventCreateWithFlags(&c->done, hipEventDisableTiming) == hipSuccess;
        if (ok) {
            // some room to grow, within what is kept
            const size_t nb = bytes > kCutKeep ? bytes : (bytes + bytes / 4 < kCutKeep ? bytes + bytes / 4 : kCutKeep);
            ok = device_alloc(&c->p, nb) == hipSuccess;
            c->bytes = ok ? nb : 0;
            if (!ok) c->p = nullptr;
        }
    }
    if (!ok) {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> lock(g_cut.m);
        c->busy = false;
        return nullptr;
    }
    c->dev = dev;
    c->st = st;
    c->used = ++g_cut.clock;
    return c->p;
}

void cut_free(void *p, hipStream_t st) {
    if (!p) return;
    std::lock_guard<std::mutex> lock(g_cut.m);
    for (CutBuf &c : g_cut.b) {
        if (!c.busy || c.p != p) continue;
        if (c.bytes > kCutKeep || hipEventRecord(c.done, st) != hipSuccess) {
            const RelaxedCapture relaxed;
            if (g_cut.holds_flags(c)) {
                (void)hipMemcpyAsync(g_cut.known, g_cut.flags, sizeof g_cut.known, hipMemcpyDeviceToHost, st);
                g_cut.flags = nullptr;
            }
            (void)hipStreamSynchronize(st);
            (void)hipFree(c.p);
            c.p = nullptr;
            c.bytes = 0;
            (void)hipGetLastError();
        }
        c.busy = false;
        return;
    }
}

}  // namespace bh

using namespace bh;

extern "C" {

int bh_init(int device) {
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count == 0) {
        set_error("no HIP device visible (%s)", hipGetErrorString(e));
        return BH_ERR_NODEVICE;
    }
    if (device < 0 || device >= count) {
        set_error("device %d out of range (%d visible)", device, count);
        return -1;
    }
    hipDeviceProp_t prop;
    BH_HIP(hipGetDeviceProperties(&prop, device));
    if (std::string(prop.gcnArchName).find("gfx950") == std::string::npos) {
        set_error("device %d is %s; this library is built for gfx950 only", device, prop.gcnArchName);
        return BH_ERR_NODEVICE;
    }
    BH_HIP(hipSetDevice(device));
    if (g_own_stream == nullptr || g_device != device) {
        // Default priority only: the library never changes stream priorities.
        BH_HIP(hipStreamCreateWithFlags(&g_own_stream, hipStreamNonBlocking));
        // library-owned control words and scratch on this device
        g_ctrl = nullptr;
        g_scratch = nullptr;
        g_scratch_bytes = 0;
        BH_HIP(hipMalloc((void **)&g_ctrl, kCtrlBytes));
        BH_HIP(hipMalloc(&g_scratch, kScratchInitial));
        g_scratch_bytes = kScratchInitial;
    }
    g_device = device;
    // the no-allocation entry point's scratch address on this device; a
    // failure is recorded there and reported by that entry point only
    (void)noalloc_setup(device);
    return BH_OK;
}

int bh_device_count(int *count) {
    BH_ARG(count != nullptr, 1);
    hipError_t e = hipGetDeviceCount(count);
    if (e != hipSuccess) *count = 0;
    return BH_OK;
}

const char *bh_last_error(void) { return g_err; }

int bh_malloc(void **dptr, size_t bytes) {
    BH_ARG(dptr != nullptr, 1);
    int st = ensure_init();
    if (st) return st;
    *dptr = nullptr;
    if (bytes == 0) return BH_OK;
    BH_HIP((hipError_t)g_blocks.take(dptr, bytes));
    return BH_OK;
}

int bh_free(void *dptr) {
    if (dptr == nullptr) return BH_OK;
    BH_HIP((hipError_t)g_blocks.give(dptr));
    return BH_OK;
}

int bh_trim(void) {
    release_kept();
    return BH_OK;
}

int bh_cut_verdict(int *verdict_host, int *tries_host) {
    BH_ARG(verdict_host != nullptr, 1);
    std::lock_guard<std::mutex> lock(g_cut.m);
    *verdict_host = 0;
    if (tries_host) *tries_host = g_cut.tries;
    if (g_cut.tries == 0) return BH_OK;
    if (g_cut.flags) {
        BH_HIP(hipMemcpyAsync(g_cut.known, g_cut.flags, sizeof g_cut.known, hipMemcpyDeviceToHost, g_cut.flags_st));
        BH_HIP(hipStreamSynchronize(g_cut.flags_st));
    }
    *verdict_host = g_cut.known[0] ? 2 : (g_cut.known[1] ? 3 : 1);
    return BH_OK;
}

int bh_memcpy_htod(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return BH_OK;
    int st = ensure_init();
    if (st) return st;
    BH_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream()));
    BH_HIP(hipStreamSynchronize(stream()));
    return BH_OK;
}

int bh_memcpy_dtoh(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return BH_OK;
    int st = ensure_init();
    if (st) return st;
    BH_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream()));
    BH_HIP(hipStreamSynchronize(stream()));
    return BH_OK;
}

int bh_memcpy_dtod(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return BH_OK;
    int st = ensure_init();
    if (st) return st;
    BH_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, stream()));
    return BH_OK;
}

int bh_memset(void *dptr, int value, size_t bytes) {
    if (bytes == 0) return BH_OK;
    int st = ensure_init();
    if (st) return st;
    BH_HIP(hipMemsetAsync(dptr, value, bytes, stream()));
    return BH_OK;
}

int bh_sync(void) {
    int st = ensure_init();
    if (st) return st;
    BH_HIP(hipStreamSynchronize(stream()));
    return BH_OK;
}

int bh_set_stream(void *s) {
    g_user_stream = (hipStream_t)s;
    return BH_OK;
}

void *bh_get_stream(void) { return (void *)stream(); }

int bh_event_create(void **ev) {
    BH_ARG(ev != nullptr, 1);
    int st = ensure_init();
    if (st) return st;
    hipEvent_t e;
    BH_HIP(hipEventCreate(&e));
    *ev = (void *)e;
    return BH_OK;
}

int bh_event_record(void *ev) {
    BH_HIP(hipEventRecord((hipEvent_t)ev, stream()));
    return BH_OK;
}

int bh_event_elapsed_ms(void *start, void *stop, float *ms) {
    BH_HIP(hipEventSynchronize((hipEvent_t)stop));
    BH_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
    return BH_OK;
}

int bh_event_destroy(void *ev) {
    if (ev) BH_HIP(hipEventDestroy((hipEvent_t)ev));
    return BH_OK;
}

}  // extern "C"
