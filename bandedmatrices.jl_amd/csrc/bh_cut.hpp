// bh_cut.hpp -- a band recurrence cut into overlapping blocks that run at once.
//
// Band factorisations and solves are chains: step j needs what step j-1 left
// in a window of the band's width, so one system keeps one workgroup (often
// one wave) busy and the rest of the chip idle.  On matrices whose diagonal
// dominates, that window forgets where the chain began: run from a wrong
// state (none of the earlier steps), it reaches not only the same values to
// rounding but the same bits after some 12 (FP64) or 8 (FP32) bandwidths --
// an entry that differs in its last bit moves the entries it touches by far
// less than half a bit of theirs.  So the n steps are cut into p blocks of L
// steps; every block starts W steps early from the bare matrix, all blocks
// run at once, and then the outcome is CHECKED: a block's factor columns (or
// window) at its end must equal, bit for bit, what the next block computed
// for the same steps before its own began.  The first block starts where the
// chain starts, so equality at every seam makes every block's result the
// sequential chain's, bit for bit.  If a seam differs nothing has been
// written to the caller's arrays yet and the sequential kernel does the work:
// launched behind the blocks with the verdict as its condition where the call
// waits for nothing (tbsv, gbtrs, gbtrs_blocked: a refused matrix pays 11-25 us
// of gate and empty launches), by the host, which learns the verdicts on the
// way, where it waits anyway (gbtrf, pbtrf, gbtrs_part: 15-20 us).
//
// The check decides the result; the gate only decides whether trying is worth
// its time (it samples columns for diagonal dominance: without it a matrix
// that needs its pivots would pay for blocks that never agree).
#pragma once
#include "bh_common.hpp"

namespace bh {

// Device memory for one call on this thread's buffer for the stream, used in the
// stream's order until cut_free: safe with any number of streams and threads.
// A thread keeps at most four buffers of kCutKeep bytes and frees them when it
// ends; larger ones go back at once.  nullptr when there is none (or more
// than kCutMax is asked for, or the stream is being captured): the caller
// takes its sequential path.
constexpr size_t kCutKeep = size_t(2) << 30;
constexpr size_t kCutMax = size_t(8) << 30;
void *cut_alloc(size_t bytes, hipStream_t st);
void cut_free(void *p, hipStream_t st);
// For a caller that waits for a verdict before it goes on: kCutWords words of
// this thread's pinned host memory, -1 each, into which kernels write values
// >= 0 (nullptr: none to be had), and a wait for one of them: its value, or -1
// when the stream has ended without it.  (A wait through a copy to the host
// left the device idle for 50 us before the next kernel, through an event some
// 15; the word is there in a few.)
constexpr int kCutWords = 4;
int *cut_host_words();
int cut_poll(const int *word, hipStream_t st);
// False when the environment says BANDEDHIP_CUT=off or a caller that may not
// allocate has switched it off for this thread.
bool cut_enabled();
// For bh_cut_verdict: a call that can run by blocks begins (nothing tried yet);
// blocks are launched whose verdict will stand in flags, in a buffer of cut_alloc.
void cut_begin();
void cut_note(const int *flags, hipStream_t st);
struct CutOff {  // no cutting on this thread while one of these lives
    CutOff();
    ~CutOff();
};

struct CutGeom {
    int n, L, W, p;
    __host__ __device__ int own(int i) const { return i * L; }
    __host__ __device__ int start(int i) const { return i * L > W ? i * L - W : 0; }
    __host__ __device__ int end(int i) const { return (i + 1) * L < n ? (i + 1) * L : n; }
    __host__ __device__ int span() const { return L + W; }  // most steps of a block
};

// flags[0]: nonzero when the gate found the matrix not worth cutting;
// flags[1]: nonzero when a seam differed or a block met a zero pivot.
__device__ __forceinline__ bool cut_closed(const int *flags) { return __hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0; }
__device__ __forceinline__ bool cut_failed(const int *flags) {
    return cut_closed(flags) || __hip_atomic_load(flags + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

// a word of the host's
__device__ __forceinline__ void cut_tell(int *word, int v) {
    if (word) __hip_atomic_store(word, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ bool cut_differ(double a, double b) {
    return __builtin_bit_cast(unsigned long long, a) != __builtin_bit_cast(unsigned long long, b);
}
__device__ __forceinline__ bool cut_differ(float a, float b) {
    return __builtin_bit_cast(unsigned, a) != __builtin_bit_cast(unsigned, b);
}

// One factorisation cut into blocks: block i factors columns start(i) ..
// end(i)-1 and the rows they reach, in a copy of its own (ld = H = 2kl+ku+1),
// as a system of its own.  g.p == 0: not cut (with flags: the sequential kernel,
// launched behind the gate, which runs only if that is closed).
template <typename T>
struct LuCut {
    CutGeom g;
    const int *flags;
    T *ab;      // p copies of span() columns
    i64 *ipiv;  // p runs of span() pivots, 1-based within the block
    i64 *info;  // two words per block
    int H, kl;
    __device__ __forceinline__ T *block_ab(int i) const { return ab + (i64)i * g.span() * H; }
    __device__ __forceinline__ int cols(int i) const { return g.end(i) - g.start(i); }
    __device__ __forceinline__ int rows(int i) const {
        const int e = g.end(i) + kl;
        return (e < g.n ? e : g.n) - g.start(i);
    }
};

// The blocks of a one-lane-per-block Cholesky (bh_pbtrf_lane.hip).
struct PbLane {
    int p, L, W;  // blocks, own columns, lead-in
};

// Gate: 256 columns spread over the matrix, 16 lanes to a column (64 columns,
// a wave to each, where they are longer than 64 entries: 42 -> 19 us at
// 385 and 129 entries); closed when more than a quarter of them have num/4 times the sum of |a| off the
// diagonal above |a_jj|.  One workgroup, so it writes both flags itself (and the
// first one to a word of the host's, where there is one, and zeroes the caller's
// two info words: a fill in front of the sequential kernel is a launch more).
// rate > 0 (a symmetric matrix of which s1 holds one triangle): closed also
// when the mean over the sampled columns of
//     -sum over the stored entries at distance t of s^t a_t (z^t + z^-t) / a_jj,  z = 2^-rate,
// is above 1 for s = 1 or s = -1.  A constant band with those coefficients
// forgets by the factor z per step (twice per step in its factorisation) where
// that sum is 1, in the mode that is constant or alternates; above it, too
// slowly for the lead-in.  Coefficients of random signs average out, as they do
// in the chain.  Dominance alone does not tell: the second difference (2, -1)
// and the five-point Laplacian (4, -1, -1) are at twice the sum of the stored
// half, and never agree; they stand at 1.02 to 1.35 here (kd = 1 .. 64, FP32
// and FP64).  Random, constant and Laplacian bands over diagonals of 1 to 2
// times the other entries, simulated: what the test closes never agrees within
// the lead-in; of what it leaves open, wide Laplacians at 1.25 to 3 times
// dominance (kd = 64) do not agree either and pay for the trial.
//
// A set of entries of a column: rows r0 .. r0+h-1 of the band array, the
// diagonal in row d (with `unit` it counts as 1); h = 0: no second set.
struct CutSet {
    int r0, h, d, unit;
};
template <typename T>
__global__ void __launch_bounds__(1024) cut_gate(const T *__restrict__ a, i64 ld, int n, CutSet s1, CutSet s2, int num,
                                                 float rate, int *flags, int *host, i64 *info) {
    __shared__ int weak[2];
    __shared__ float part[2][16];
    if (threadIdx.x < 2) weak[threadIdx.x] = 0;
    __syncthreads();
    const int lanes = s1.h > 64 ? 64 : 16, cols = 1024 / lanes, samples = 4 * cols;
    const int g = threadIdx.x / lanes, q = threadIdx.x & (lanes - 1);
    int m1 = 0, m2 = 0;
    auto strong = [&](const T *col, const CutSet &s) {
        T t = T(0);
        for (int r = q; r < s.h; r += lanes) t += (s.r0 + r == s.d) ? T(0) : dabs(col[s.r0 + r]);
        for (int off = lanes / 2; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
        return T(4) * (s.unit ? T(1) : dabs(col[s.d])) >= T(num) * t;
    };
    // per lane, over its entries of all its columns
    float mean[2] = {0.0f, 0.0f};
    auto coherent = [&](const T *col, i64 c, int r, T w) {  // slots outside the matrix hold anything
        const int dist = s1.r0 + r - s1.d;
        if (dist == 0 || c + dist < 0 || c + dist >= n) return;
        const float t = (float)(col[s1.r0 + r] * w / col[s1.d]);
        mean[0] -= t;
        mean[1] -= dist & 1 ? -t : t;
    };
    const T *col[4];
    i64 cs[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        // the golden section spreads the samples evenly without a stride, which a
        // grid's rows could be in step with
        cs[it] = (i64)(((unsigned long long)((unsigned)(cols * it + g + 1) * 2654435769u) * (unsigned)n) >> 32);
        col[it] = a + cs[it] * ld;
    }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        m1 += !strong(col[it], s1);
        if (s2.h) m2 += !strong(col[it], s2);
    }
    if (rate > 0.0f)
        for (int r = q; r < s1.h; r += lanes) {
            const float z = exp2f(rate * (float)(s1.r0 + r - s1.d));
            const T w = T(z + 1.0f / z);
#pragma unroll
            for (int it = 0; it < 4; ++it) coherent(col[it], cs[it], r, w);
        }
    for (int off = 32; off > 0; off >>= 1) {
        mean[0] += __shfl_xor(mean[0], off, 64);
        mean[1] += __shfl_xor(mean[1], off, 64);
    }
    if (q == 0) {
        atomicAdd(&weak[0], m1);
        atomicAdd(&weak[1], m2);
    }
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = mean[0];
        part[1][threadIdx.x >> 6] = mean[1];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float t0 = 0.0f, t1 = 0.0f;
        for (int i = 0; i < 16; ++i) {
            t0 += part[0][i];
            t1 += part[1][i];
        }
        const int closed =
            weak[0] > samples / 4 || weak[1] > samples / 4 || !(t0 <= (float)samples) || !(t1 <= (float)samples);
        flags[0] = closed;
        flags[1] = 0;
        if (info) info[0] = info[1] = 0;
        cut_tell(host, closed);
    }
}

// The gate's rate for a lead-in of W steps: the chain forgets twice the rate's
// bits a step, and all but the last few of the type's must be gone after W.
template <typename T>
inline float cut_rate(i64 W) {
    return (sizeof(T) == 8 ? 48.0f : 24.0f) / (2.0f * (float)W);
}

// ---------------------------------------------------------------- solves
// A substitution sweep cut into blocks: the state is the wave's window of the
// vector (64 NR entries in registers), steps go in groups of 64.  Every block
// writes its window down when its own groups begin (slot 0) and when they end
// (slot 1); slot 1 of a block must equal slot 0 of the next.
template <typename T>
struct SweepCut {
    CutGeom g;  // in groups, along the sweep; g.p == 0: the whole sweep (with flags: only if the blocks failed)
    const int *flags;
    T *snap;
    __device__ __forceinline__ T *at(int blk, int which, int cnt) const {
        return snap + (((i64)blk * gridDim.x + blockIdx.x) * 2 + which) * cnt;
    }
};

// The memory of a solve by blocks alone (nullptr: it is not to be had that way)
// and its verdict, freed by whoever asked for it.
struct RingCutWs {
    void *ws = nullptr;
    int *flags = nullptr;
    int *host = nullptr;  // [0]: whether the gate is closed; [1]: whether the blocks failed; two more for the caller
};

// cnt entries per window; grid (p - 1, nrhs)
template <typename T>
__global__ void __launch_bounds__(256) sweep_check(const T *__restrict__ snap, int cnt, int *flags) {
    if (cut_closed(flags)) return;
    const T *e = snap + (((i64)blockIdx.x * gridDim.y + blockIdx.y) * 2 + 1) * cnt;
    const T *s = snap + (((i64)(blockIdx.x + 1) * gridDim.y + blockIdx.y) * 2) * cnt;
    bool bad = false;
#pragma unroll 4
    for (int i = threadIdx.x; i < cnt; i += 256) bad |= cut_differ(e[i], s[i]);
    if (__syncthreads_or(bad) && threadIdx.x == 0) atomicOr(flags + 1, 1);
}

// the blocks' results (n x nrhs, contiguous) to the caller's vectors; host: told whether they failed
template <typename T>
__global__ void __launch_bounds__(256) sweep_commit(int n, const T *__restrict__ y, T *__restrict__ x, int incx,
                                                    i64 ldx, const int *flags, int *host) {
    const bool failed = cut_failed(flags);
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) cut_tell(host, failed);
    if (failed) return;
    const i64 i = (i64)blockIdx.x * 256 + threadIdx.x;
    if (i < n) x[(i64)blockIdx.y * ldx + i * incx] = y[(i64)blockIdx.y * n + i];
}

// Groups of a sweep over n steps with bandwidth k, nrhs vectors.  Lead-in:
// measured on the factors of dominant random matrices the windows agree after
// 12-18 k steps in FP64 (k = 4 .. 64; 23 k at k = 2) and 7-10 k in FP32; 20 k
// and 10 k, with nw whole groups more for the window itself (64 steps and up,
// which at k = 2 is another 32 k).  Factors of constant sparse bands forget more
// slowly (a five-point operator at 1.25 to 1.5 times dominance: 28-41 k): those
// differ and pay for the trial.  Own groups: about 2048 waves (two per SIMD) over all
// vectors, and not under half the lead-in, which every block repeats.
template <typename T>
inline CutGeom sweep_geom(i64 n, i64 k, i64 nrhs, i64 nw) {
    const i64 G = cdiv(n, 64), W = cdiv((sizeof(T) == 8 ? 20 : 10) * k, 64) + nw;
    const i64 L = imax(cdiv(G, imax(1, 2048 / nrhs)), (W + 1) / 2);
    CutGeom g{(int)G, (int)L, (int)W, (int)cdiv(G, L)};
    if (3 * (L + W) > G || nrhs > 65535) g.p = 0;
    return g;
}

}  // namespace bh
