// bh_pbtrf_lane.hip -- band Cholesky of an upper triangle by blocks, one lane
// per block, for kd <= 8 (bh_pbtrf.hip launches it for dominant matrices).
//
// The workgroup kernel pays two barriers a column for kd(kd+3)/2 operations.
// Here a lane factors its own block, and what is live of it sits in registers: with R =
// kd+1, entry (i, j), i <= j <= i+kd, in register [i mod R][j mod R].  The
// active triangle and the finished entries of the columns still open fill
// that square exactly: column j is complete at step j, goes out as it lies in
// storage, and column j+R takes its place.  xPBTF2's operations in its order
// (reciprocal-scaled row, rank-1 update skipping zero entries): the same bits.
// n = 65536, kd = 8, FP64: 0.32 -> 0.13 ms; a step takes 0.7 us (root, division,
// 36 fused updates and their zero tests, one wave issuing them).
#include "bh_common.hpp"
#include "bh_cut.hpp"

namespace bh {

namespace {

template <int I>
struct PK {
    static constexpr int value = I;
};
template <int N>
struct PLUnroll {
    template <class F>
    __device__ __forceinline__ static void run(F &&f) {
        PLUnroll<N - 1>::run(f);
        f(PK<N - 1>{});
    }
};
template <>
struct PLUnroll<0> {
    template <class F>
    __device__ __forceinline__ static void run(F &&) {}
};
__device__ __forceinline__ __amdgpu_buffer_rsrc_t pl_rsrc(const void *p, i64 bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ double pl_ld(__amdgpu_buffer_rsrc_t r, int off, double) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ float pl_ld(__amdgpu_buffer_rsrc_t r, int off, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ void pl_st(__amdgpu_buffer_rsrc_t r, int off, double v) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, off, 0, 0);
}
__device__ __forceinline__ void pl_st(__amdgpu_buffer_rsrc_t r, int off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
}
__device__ __forceinline__ double pl_sqrt(double x) { return __builtin_sqrt(x); }
__device__ __forceinline__ float pl_sqrt(float x) { return __builtin_sqrtf(x); }

// Own columns go to out (n columns of ld K+1); the K columns before a block's
// own and the K last of its own go to seam (two sets of K x (K+1) entries per
// block, lane-interleaved) for the check.  Columns before the matrix or past its
// end run as the identity's.
template <typename T, int K>
__global__ void __launch_bounds__(64) pbtrf_lane(int n, const T *__restrict__ ab, i64 lda, T *__restrict__ out, int L, int W,
                                                 int p, T *__restrict__ seam, int *flags) {
    constexpr int R = K + 1, SZ = (int)sizeof(T), OOB = 0x7ff00000;
    constexpr int PD = sizeof(T) == 8 && K > 6 ? 1 : 2;  // columns prefetched, in units of R
    if (cut_closed(flags)) return;
    const int blk = blockIdx.x * 64 + (int)__lane_id();
    const __amdgpu_buffer_rsrc_t ra = pl_rsrc(ab, ((i64)(n - 1) * lda + R) * SZ);
    const __amdgpu_buffer_rsrc_t ro = pl_rsrc(out, (i64)n * R * SZ);
    const int own = blk * L, c0 = own - W, past = own + L < n ? own + L : n;
    auto in = [&](int c) { return c >= 0 && c < n && blk < p; };
    // column c: entry (c - K + r, c) in row r.  (Rows before the block's first
    // column are never used; in the first wave, whose blocks begin before the
    // matrix, the slots above row 0 read as zeros.)
    auto column = [&](int c, T (&v)[R]) {
        const int off = in(c) ? c * (int)lda * SZ : OOB;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = pl_ld(ra, off + r * SZ, T());
        v[K] = in(c) ? v[K] : T(1);
        if (blockIdx.x == 0) {
#pragma unroll
            for (int r = 0; r < K; ++r) v[r] = c < K - r ? T(0) : v[r];
        }
    };
    T A[R][R];  // [i mod R][j mod R], indexes relative to c0
    T nx[PD * R][R];
    PLUnroll<R>::run([&](auto jc) {
        constexpr int j = decltype(jc)::value;  // columns c0 .. c0+K
        T v[R];
        column(c0 + j, v);
        PLUnroll<R>::run([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            A[(j - K + r + R) % R][j] = v[r];
        });
    });
    PLUnroll<PD * R>::run([&](auto jc) { column(c0 + R + decltype(jc)::value, nx[decltype(jc)::value]); });
    bool bad = false;
    auto block = [&](int s0, auto half) {
        PLUnroll<R>::run([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            const int c = c0 + s0 + s;
            const T a = A[s][s];
            bad |= a <= T(0);
            const T root = pl_sqrt(a);
            A[s][s] = root;
            const T rcp = T(1) / root;
            T v[R];
#pragma unroll
            for (int q = 1; q < R; ++q) {
                v[q] = A[s][(s + q) % R] * rcp;
                A[s][(s + q) % R] = v[q];
            }
#pragma unroll
            for (int q = 1; q < R; ++q) {
                const T tq = -v[q];
                if (v[q] != T(0)) {
#pragma unroll
                    for (int e = 1; e <= q; ++e) A[(s + e) % R][(s + q) % R] = dfma(tq, v[e], A[(s + e) % R][(s + q) % R]);
                }
            }
            // column c is complete: rows c-K .. c
            const int oo = c >= own && c < past && blk < p ? c * R * SZ : OOB;
#pragma unroll
            for (int r = 0; r < R; ++r) pl_st(ro, oo + r * SZ, A[(s - K + r + R) % R][s]);
            const int before = c - (own - K), last = c - (own + L - K);
            const bool kb = before >= 0 && before < K, kl = last >= 0 && last < K;
            if (kb || kl) {
                T *d = seam + ((i64)((kb ? 0 : K) + (kb ? before : last)) * R) * p + blk;
                if (blk < p)
#pragma unroll
                    for (int r = 0; r < R; ++r) d[(i64)r * p] = A[(s - K + r + R) % R][s];
            }
            constexpr int slot = decltype(half)::value * R + s;
#pragma unroll
            for (int r = 0; r < R; ++r) A[(s + 1 + r) % R][s] = nx[slot][r];  // column c + R, rows c+1 .. c+R
            column(c + R + PD * R, nx[slot]);
        });
    };
    for (int s0 = 0; s0 < W + L; s0 += PD * R) {  // W + L: a multiple of PD*R
        block(s0, PK<0>{});
        if constexpr (PD == 2) block(s0 + R, PK<1>{});
    }
    if (bad) atomicOr(flags + 1, 1);
}

// cnt = K (K+1) entries; the last own columns of block b against those block
// b+1 ran before its own
template <typename T>
__global__ void __launch_bounds__(256) pbtrf_lane_check(int p, int cnt, const T *__restrict__ seam, int *flags) {
    if (cut_closed(flags)) return;
    const int b = blockIdx.x * 256 + threadIdx.x;
    bool bad = false;
    if (b + 1 < p)
        for (int i = blockIdx.y; i < cnt; i += gridDim.y) bad |= cut_differ(seam[(i64)(cnt + i) * p + b], seam[(i64)i * p + b + 1]);
    if (__syncthreads_or(bad) && threadIdx.x == 0) atomicOr(flags + 1, 1);
}

template <typename T>
__global__ void __launch_bounds__(256) pbtrf_lane_commit(int n, int H, const T *__restrict__ out, T *__restrict__ ab, i64 lda,
                                                         const int *flags, int *host) {
    const bool failed = cut_failed(flags);
    if (blockIdx.x == 0 && threadIdx.x == 0) cut_tell(host, failed);
    if (failed) return;
    const i64 e = (i64)blockIdx.x * 256 + threadIdx.x;
    if (e >= (i64)n * H) return;
    const i64 c = e / H;
    const int r = (int)(e - c * H);
    if (c - H + 1 + r >= 0) ab[c * lda + r] = out[e];  // slots outside the matrix stay as they are
}

}  // namespace

// Own steps and lead-in of the blocks (p = 0: not taken): lead-in as
// pb_cut_geom's; up to 8192 lanes, at least 24 own columns each.
template <typename T>
PbLane pbtrf_lane_geom(i64 n, i64 kd, i64 ldab) {
    PbLane g{0, 0, 0};
    const i64 lim = (1ll << 31) - (1 << 24);
    if (kd < 1 || kd > 8 || n >= (1ll << 29) || ldab * n * (i64)sizeof(T) >= lim) return g;
    const i64 U = (sizeof(T) == 8 && kd > 6 ? 1 : 2) * (kd + 1);  // steps unrolled together
    const i64 W = U * cdiv((sizeof(T) == 8 ? 14 : 8) * kd + 32, U), L = U * cdiv(imax(24, cdiv(n, 8192)), U);
    if (3 * (L + W) > n) return g;
    g.p = (int)cdiv(n, L);
    g.L = (int)L;
    g.W = (int)W;
    return g;
}

// out: n x (kd+1), seam: 2 kd (kd+1) p entries.
template <typename T>
int pbtrf_lane_run(const PbLane &g, i64 n, i64 kd, T *ab, i64 ldab, T *out, T *seam, int *flags, int *host,
                   hipStream_t st) {
    const dim3 grid((unsigned)cdiv(g.p, 64));
    switch ((int)kd) {
#define BH_PL_CASE(Kv)                                                                                              \
    case Kv:                                                                                                        \
        hipLaunchKernelGGL((pbtrf_lane<T, Kv>), grid, dim3(64), 0, st, (int)n, (const T *)ab, ldab, out, g.L, g.W, g.p, \
                           seam, flags);                                                                            \
        break;
        BH_PL_CASE(1) BH_PL_CASE(2) BH_PL_CASE(3) BH_PL_CASE(4) BH_PL_CASE(5) BH_PL_CASE(6) BH_PL_CASE(7) BH_PL_CASE(8)
#undef BH_PL_CASE
        default:
            return BH_ERR_INTERNAL;
    }
    const int cnt = (int)(kd * (kd + 1));
    hipLaunchKernelGGL(pbtrf_lane_check<T>, dim3((unsigned)cdiv(g.p, 256), imin(cnt, 16)), dim3(256), 0, st, g.p, cnt,
                       (const T *)seam, flags);
    hipLaunchKernelGGL(pbtrf_lane_commit<T>, dim3((unsigned)cdiv(n * (kd + 1), 256)), dim3(256), 0, st, (int)n,
                       (int)kd + 1, (const T *)out, ab, ldab, (const int *)flags, host);
    return BH_OK;
}

template PbLane pbtrf_lane_geom<double>(i64, i64, i64);
template PbLane pbtrf_lane_geom<float>(i64, i64, i64);
template int pbtrf_lane_run<double>(const PbLane &, i64, i64, double *, i64, double *, double *, int *, int *,
                                    hipStream_t);
template int pbtrf_lane_run<float>(const PbLane &, i64, i64, float *, i64, float *, float *, int *, int *,
                                   hipStream_t);

}  // namespace bh
