// bh_tbsv_lane.hpp -- the 'N' triangular band solve by blocks with one lane per
// block (k <= 16): compiled per element type in bh_tbsv_lane_{d,s}.hip
// (BH_TL_T), called by bh_tbsv.hpp.
//
// The ring (one wave per block) issues some fifty instructions for a step's k
// useful ones.  Here 64 blocks share a wave: a lane walks its own block, the
// window of the vector in registers renamed by unrolling, one division and k
// fused updates a step in the ring's order, so the same bits.  Each lane reads its
// own columns (contiguous k+1 entries), PD steps ahead.
#pragma once
#include "bh_common.hpp"
#include "bh_cut.hpp"

namespace bh {

// The blocks of a 'N' solve; p = 0: a k or size they do not take.
struct TbsvLane {
    int p = 0, L = 0, W = 0;  // blocks, own steps, lead-in
};
TbsvLane tbsv_lane_geom(i64 n, i64 k, i64 lda, i64 incx, i64 ldx, i64 nrhs, int elem);
inline size_t tbsv_lane_bytes(const TbsvLane &g, i64 k, i64 nrhs, size_t elem) { return (size_t)2 * g.p * k * nrhs * elem; }
// Runs them (asc: lower, else upper) and their seam checks into flags; y (n x
// nrhs) takes the result, snap (tbsv_lane_bytes) the windows.
int tbsv_lane_run(const TbsvLane &g, bool asc, int n, int k, const double *a, i64 lda, const double *x, int incx, i64 ldx,
                  int nrhs, bool unit, double *y, double *snap, int *flags, hipStream_t st);
int tbsv_lane_run(const TbsvLane &g, bool asc, int n, int k, const float *a, i64 lda, const float *x, int incx, i64 ldx,
                  int nrhs, bool unit, float *y, float *snap, int *flags, hipStream_t st);

#ifdef BH_TL_T
namespace {

template <int I>
struct LK {
    static constexpr int value = I;
};
template <int N>
struct LUnroll {
    template <class F>
    __device__ __forceinline__ static void run(F &&f) {
        LUnroll<N - 1>::run(f);
        f(LK<N - 1>{});
    }
};
template <>
struct LUnroll<0> {
    template <class F>
    __device__ __forceinline__ static void run(F &&) {}
};
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tl_rsrc(const void *p, i64 bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ double tl_ld(__amdgpu_buffer_rsrc_t r, int off, double) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ float tl_ld(__amdgpu_buffer_rsrc_t r, int off, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ void tl_st(__amdgpu_buffer_rsrc_t r, int off, double v) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, off, 0, 0);
}
__device__ __forceinline__ void tl_st(__amdgpu_buffer_rsrc_t r, int off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
}

// window registers: at least k+1, at least 8 (the prefetch distance), even where it is halved
template <int K>
struct TlShape {
    static constexpr int R = K <= 7 ? 8 : K <= 10 ? K + 1 : (K + 2) / 2 * 2;
    static constexpr int PD = K <= 10 ? R : R / 2;
};

// Step c of the chain is row c (ASC) or n-1-c.  Steps before the chain or past
// its end read zeros and a unit diagonal: they leave every entry as it is.
template <typename T, int K, bool ASC>
__global__ void __launch_bounds__(64) tbsv_lane(int n, const T *__restrict__ a, i64 lda, const T *__restrict__ x, int incx,
                                                i64 ldx, int unit, T *__restrict__ y, TbsvLane g, T *__restrict__ snap,
                                                const int *flags) {
    constexpr int R = TlShape<K>::R, PD = TlShape<K>::PD;
    constexpr int SZ = (int)sizeof(T), OOB = 0x7ff00000;
    if (cut_closed(flags)) return;
    const int blk = blockIdx.x * 64 + (int)__lane_id(), rhs = blockIdx.y;
    const __amdgpu_buffer_rsrc_t ra = tl_rsrc(a, ((i64)(n - 1) * lda + K + 1) * SZ);
    const __amdgpu_buffer_rsrc_t rx = tl_rsrc(x + (i64)rhs * ldx, ((i64)(n - 1) * incx + 1) * SZ);
    const __amdgpu_buffer_rsrc_t ry = tl_rsrc(y + (i64)rhs * n, (i64)n * SZ);
    const int own = blk * g.L, c0 = own - g.W;
    const int past = own + g.L < n ? own + g.L : n;  // first chain step that is not this block's
    auto row = [&](int c) { return ASC ? c : n - 1 - c; };
    auto in = [&](int c) { return c >= 0 && c < n && blk < g.p; };
    auto xin = [&](int c) -> T { return tl_ld(rx, in(c) ? row(c) * incx * SZ : OOB, T()); };
    T w[R], f[PD][K], d[PD], bp[PD];
    auto fetch = [&](auto slotc, int c) {
        constexpr int slot = decltype(slotc)::value;
        const int off = in(c) ? row(c) * (int)lda * SZ : OOB;
#pragma unroll
        for (int t = 1; t <= K; ++t) f[slot][t - 1] = tl_ld(ra, off + (ASC ? t : K - t) * SZ, T());
        const T dv = tl_ld(ra, off + (ASC ? 0 : K) * SZ, T());
        d[slot] = in(c) && !unit ? dv : T(1);
        bp[slot] = xin(c + R);  // the entry that takes this step's register
    };
#pragma unroll
    for (int i = 0; i < R; ++i) w[i] = xin(c0 + i);
    LUnroll<PD>::run([&](auto sc) { fetch(sc, c0 + decltype(sc)::value); });
    auto keep = [&](int which) {
        if (blk < g.p) {
#pragma unroll
            for (int i = 0; i < K; ++i) snap[(((i64)rhs * 2 + which) * K + i) * g.p + blk] = w[i];
        }
    };
    const int steps = g.W + g.L;  // multiples of R
    for (int s0 = 0; s0 < steps; s0 += R) {
        if (s0 == g.W) keep(0);
        LUnroll<R>::run([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            constexpr int slot = s % PD;
            const int c = c0 + s0 + s;
            const T xj = w[s] / d[slot];
            tl_st(ry, c >= own && c < past ? row(c) * SZ : OOB, xj);
            const T nx = -xj;
#pragma unroll
            for (int t = 1; t <= K; ++t) w[(s + t) % R] = dfma(f[slot][t - 1], nx, w[(s + t) % R]);
            w[s] = bp[slot];
            fetch(LK<slot>{}, c + PD);
        });
    }
    keep(1);
}

template <typename T>
__global__ void __launch_bounds__(256) tbsv_lane_check(int p, int k, const T *__restrict__ snap, int *flags) {
    if (cut_closed(flags)) return;
    const int b = blockIdx.x * 256 + threadIdx.x;
    bool bad = false;
    if (b + 1 < p) {
        const T *s = snap + (i64)blockIdx.y * 2 * k * p;
        for (int i = 0; i < k; ++i) bad |= cut_differ(s[(i64)(k + i) * p + b], s[(i64)i * p + b + 1]);
    }
    if (__syncthreads_or(bad) && threadIdx.x == 0) atomicOr(flags + 1, 1);
}

}  // namespace

int tbsv_lane_run(const TbsvLane &g, bool asc, int n, int k, const BH_TL_T *a, i64 lda, const BH_TL_T *x, int incx, i64 ldx,
                  int nrhs, bool unit, BH_TL_T *y, BH_TL_T *snap, int *flags, hipStream_t st) {
    using T = BH_TL_T;
    const dim3 grid((unsigned)cdiv(g.p, 64), nrhs);
    switch (k) {
#define BH_TL_CASE(Kv)                                                                                              \
    case Kv:                                                                                                        \
        if (asc)                                                                                                    \
            hipLaunchKernelGGL((tbsv_lane<T, Kv, true>), grid, dim3(64), 0, st, n, a, lda, x, incx, ldx, (int)unit, y, \
                               g, snap, (const int *)flags);                                                        \
        else                                                                                                        \
            hipLaunchKernelGGL((tbsv_lane<T, Kv, false>), grid, dim3(64), 0, st, n, a, lda, x, incx, ldx, (int)unit, y, \
                               g, snap, (const int *)flags);                                                        \
        break;
        BH_TL_CASE(1) BH_TL_CASE(2) BH_TL_CASE(3) BH_TL_CASE(4) BH_TL_CASE(5) BH_TL_CASE(6) BH_TL_CASE(7) BH_TL_CASE(8)
        BH_TL_CASE(9) BH_TL_CASE(10) BH_TL_CASE(11) BH_TL_CASE(12) BH_TL_CASE(13) BH_TL_CASE(14) BH_TL_CASE(15)
        BH_TL_CASE(16)
#undef BH_TL_CASE
        default:
            return BH_ERR_INTERNAL;
    }
    hipLaunchKernelGGL(tbsv_lane_check<T>, dim3((unsigned)cdiv(g.p, 256), nrhs), dim3(256), 0, st, g.p, k,
                       (const T *)snap, flags);
    return BH_OK;
}
#endif  // BH_TL_T

}  // namespace bh
