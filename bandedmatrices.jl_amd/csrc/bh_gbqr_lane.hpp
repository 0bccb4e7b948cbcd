// bh_gbqr_lane.hpp -- banded Householder QR of narrow bands (l <= 7) and the
// application of its Q', one wave, the band's subdiagonal count fixed at
// compile time.  Instantiated per element type in bh_gbqr_lane_{d,s}.hip
// (BH_QL_T); bh_gbqr.hip calls the launchers.
//
// The arithmetic is gbqrf_wave's and gbqr_apply_wave's (bh_gbqr.hip), bit for
// bit: the reference's sequential sums in the factor, the wave's pairwise sum
// in the application.
#pragma once
#include "bh_common.hpp"

#include <type_traits>

namespace bh {

// -1: a band, size or leading dimension these do not take.
int lane_gbqrf_launch(i64 m, i64 n, i64 l, i64 u, double *D, i64 ldd, double *tau, hipStream_t st);
int lane_gbqrf_launch(i64 m, i64 n, i64 l, i64 u, float *D, i64 ldd, float *tau, hipStream_t st);
int lane_qtb_launch(i64 m, i64 n, i64 l, i64 u, const double *D, i64 ldd, const double *tau, i64 nrhs, double *B,
                    i64 ldb, hipStream_t st);
int lane_qtb_launch(i64 m, i64 n, i64 l, i64 u, const float *D, i64 ldd, const float *tau, i64 nrhs, float *B, i64 ldb,
                    hipStream_t st);

#ifdef BH_QL_T
namespace {

template <int K>
struct QK {
    static constexpr int value = K;
};
template <int N>
struct QUnroll {
    template <class F>
    __device__ __forceinline__ static void run(F &&f) {
        QUnroll<N - 1>::run(f);
        f(QK<N - 1>{});
    }
};
template <>
struct QUnroll<0> {
    template <class F>
    __device__ __forceinline__ static void run(F &&) {}
};

__device__ __forceinline__ int ql_min(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ql_rsrc(const void *p, i64 bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
typedef unsigned ql_v2u __attribute__((ext_vector_type(2)));
// off: the lane's byte offset (past the end: nothing moves), uni: a uniform one
__device__ __forceinline__ double ql_ld(__amdgpu_buffer_rsrc_t r, int off, int uni, double) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, uni, 0));
}
__device__ __forceinline__ float ql_ld(__amdgpu_buffer_rsrc_t r, int off, int uni, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, uni, 0));
}
__device__ __forceinline__ void ql_st(__amdgpu_buffer_rsrc_t r, int off, int uni, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(ql_v2u, v), r, off, uni, 0);
}
__device__ __forceinline__ void ql_st(__amdgpu_buffer_rsrc_t r, int off, int uni, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, uni, 0);
}
__device__ __forceinline__ double ql_sqrt(double x) { return __builtin_sqrt(x); }
__device__ __forceinline__ float ql_sqrt(float x) { return __builtin_sqrtf(x); }
__device__ __forceinline__ double ql_copysign(double a, double b) { return __builtin_copysign(a, b); }
__device__ __forceinline__ float ql_copysign(float a, float b) { return __builtin_copysignf(a, b); }

// v with lane I replaced by the uniform x (unrolled callers pass a constant)
template <int I>
__device__ __forceinline__ float ql_put1(float v, float x) {
    unsigned r = __builtin_bit_cast(unsigned, v);
    asm("v_writelane_b32 %0, %1, %2" : "+v"(r) : "s"(__builtin_bit_cast(unsigned, x)), "n"(I));
    return __builtin_bit_cast(float, r);
}
template <int I>
__device__ __forceinline__ double ql_put1(double v, double x) {
    const ql_v2u a = __builtin_bit_cast(ql_v2u, v), b = __builtin_bit_cast(ql_v2u, x);
    unsigned lo = a[0], hi = a[1];
    asm("v_writelane_b32 %0, %2, %4\n\tv_writelane_b32 %1, %3, %4"
        : "+v"(lo), "+v"(hi)
        : "s"(b[0]), "s"(b[1]), "n"(I));
    return __builtin_bit_cast(double, (ql_v2u){lo, hi});
}

// Factor.  Lane c mod 64 holds column c, rows k .. k+L in registers that
// rotate with the unrolled steps (row i of step s in register (i + s) mod
// (L+1)), so nothing moves between registers; a row enters every lane's
// column one step before it can be needed, U steps ahead of its use.  The
// column is read into scalar operands once and its L+1 divisions are done as
// one, in L+1 lanes.  n = 100000, (4,4), FP64: 1.02 -> 0.39 us a column; what
// bounds it is the chain norm -> square root -> division -> v'y -> update, some
// forty dependent FP64 operations (a division sequence per entry, 34
// instructions more, took 0.40).
template <typename T, int L>
__global__ void __launch_bounds__(64) gbqrf_lane(int m, int n, int u, T *D, i64 ld, T *tau) {
    constexpr int R = L + 1;
    constexpr int U = R * ((11 + R) / R);  // steps per unrolled block, a multiple of R
    constexpr int SZ = (int)sizeof(T);
    const int lane = (int)__lane_id();
    const int mn = ql_min(m, n), ncols = ql_min(m - 1, n);
    for (int k = ncols + lane; k < mn; k += 64) tau[k] = T(0);
    if (ncols <= 0) return;
    const __amdgpu_buffer_rsrc_t rD = ql_rsrc(D, ld * (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rt = ql_rsrc(tau, (i64)mn * SZ);
    const int dstep = (int)(ld - 1) * SZ, ldb = (int)ld * SZ, ub = u * SZ;
    // row r0+L of the lane's column in the window that begins at r0 (columns
    // r0 .. r0+u+L: up to u past the row)
    auto enter = [&](int r0) -> T {
        const int d = (lane - r0) & 63;
        const int lim = r0 + L < m ? ql_min(u + L, n - 1 - r0) : -1;
        return ql_ld(rD, d <= lim ? (int)__umul24(d, dstep) : -1, r0 * ldb + ub + L * SZ, T());
    };
    T y[R], pre[U];
#pragma unroll
    for (int i = 0; i < R; ++i) {  // rows 0 .. L of the first window
        const bool ok = i < m && lane < n && lane - i <= u && i - lane <= L;
        y[i] = ql_ld(rD, ok ? lane * ldb + ub + (i - lane) * SZ : -1, 0, T());
    }
    QUnroll<U>::run([&](auto sc) { pre[decltype(sc)::value] = enter(decltype(sc)::value + 1); });
    T tk = T(0);  // tau of the block's steps, step s in lane s
    int k0 = 0;
    auto step = [&](auto sc, auto tc) {
        constexpr int s = decltype(sc)::value;
        constexpr bool TAIL = decltype(tc)::value;
        const int k = k0 + s;
        if (TAIL && k >= ncols) return;
        const int own = k & 63, len = TAIL ? ql_min(R, m - k) : R;
        auto reg = [](int i) { return (i + s) % R; };
        // column k, uniform
        T x[R];
#pragma unroll
        for (int i = 0; i < R; ++i) x[i] = lane_read(y[reg(i)], own);
        T nrm = x[0] * x[0];
#pragma unroll
        for (int i = 1; i < R; ++i)
            if (!TAIL || i < len) nrm = nrm + x[i] * x[i];
        const bool some = nrm != T(0);
        const T nu = ql_copysign(ql_sqrt(nrm), x[0]);
        const T xi1 = x[0] + nu;
        // the divisions x_i / xi1 (lane i) and xi1 / nu = tau (lane 0) as one
        T num = xi1;
        QUnroll<L>::run([&](auto ic) {
            constexpr int i = decltype(ic)::value + 1;
            num = ql_put1<i>(num, x[i]);
        });
        const T quo = num / (lane == 0 ? nu : xi1);
        const T ts = some ? lane_read(quo, 0) : T(0);
        T vs[R];
#pragma unroll
        for (int i = 1; i < R; ++i) vs[i] = some && (!TAIL || i < len) ? lane_read(quo, i) : x[i];
        tk = lane == s ? ts : tk;
        // applied to columns k+1 .. k+u
        const int d = (lane - k) & 63;
        const int last = ql_min(u, n - 1 - k);
        const bool app = (unsigned)(d - 1) < (unsigned)last;
        T w = y[reg(0)];
#pragma unroll
        for (int i = 1; i < R; ++i)
            if (!TAIL || i < len) w = w + vs[i] * y[reg(i)];
        w = ts * w;
        const T r0 = app ? y[reg(0)] - w : (some ? -nu : y[reg(0)]);  // lane own: R's diagonal
        // outputs: row k of the window's columns, the reflector from lanes 1 .. L
        const int rowb = k * ldb + ub;
        ql_st(rD, d <= last ? (int)__umul24(d, dstep) : -1, rowb, r0);
        // (a column whose squares sum to zero stands as the updates left it)
        ql_st(rD, lane >= 1 && lane < len ? lane * SZ : -1, rowb, some ? quo : num);
#pragma unroll
        for (int i = 1; i < R; ++i)
            if (!TAIL || i < len) {
                const T z = y[reg(i)] - vs[i] * w;
                y[reg(i)] = app ? z : y[reg(i)];
            }
        y[reg(0)] = pre[s];
        pre[s] = enter(k + U + 1);
    };
    auto put_tau = [&] { ql_st(rt, (lane < U && k0 + lane < ncols) ? (k0 + lane) * SZ : -1, 0, tk); };
    const int kmain = ql_min(ncols, m - L);  // steps before it have all L+1 rows
    for (; k0 + U <= kmain; k0 += U) {
        QUnroll<U>::run([&](auto sc) { step(sc, std::false_type{}); });
        put_tau();
    }
    for (; k0 < ncols; k0 += U) {
        QUnroll<U>::run([&](auto sc) { step(sc, std::true_type{}); });
        put_tau();
    }
    // Row ncols (if < m) of the columns still in the window is final too: no
    // later reflector touches it.  The last block may have ended early, so
    // its register depends on where.
    {
        const int r = ncols, d = (lane - r) & 63;
        const int at = (ncols - (k0 - U)) % R;
        T z = y[0];
#pragma unroll
        for (int i = 1; i < R; ++i) z = at == i ? y[i] : z;
        ql_st(rD, (r < m && d <= ql_min(u, n - 1 - r)) ? (int)__umul24(d, dstep) : -1, r * ldb + ub, z);
    }
}

// B <- Q'B.  Reflectors are uniform over the wave: a block's are loaded a
// block ahead, one step to a lane, and read into scalar operands, so no step
// waits for memory (a window of loads U steps ahead did: 0.29 us a step) and
// no step crosses lanes.  ONE: one right-hand side, uniform as well (blocks of
// it loaded and stored across the lanes); otherwise one lane per right-hand
// side.  v'b is summed as the wave sum of gbqr_apply_wave adds its first eight
// lanes.  n = 100000, (4,4), FP64, one right-hand side: 0.49 -> 0.071 us a
// reflector.
template <typename T, int L, bool ONE>
__global__ void __launch_bounds__(64) qtb_lane(int m, int u, const T *D, i64 ld, i64 ncol, const T *tau, int kmax, T *B,
                                               i64 ldb, int nrhs) {
    constexpr int R = L + 1;
    constexpr int U = R * ((ONE ? 64 : 32) / R);  // steps of a block
    constexpr int SZ = (int)sizeof(T);
    const int lane = (int)__lane_id(), c = blockIdx.x * 64 + lane;
    const __amdgpu_buffer_rsrc_t rD = ql_rsrc(D, ld * ncol * SZ);
    const __amdgpu_buffer_rsrc_t rt = ql_rsrc(tau, (i64)kmax * SZ);
    const __amdgpu_buffer_rsrc_t rB = ql_rsrc(B, ldb * (i64)nrhs * SZ);
    const int colb = c < nrhs ? c * (int)ldb * SZ : -1;
    const int ldD = (int)ld * SZ, ub = u * SZ;
    T w[R], xb[R], tb, bb = T(0), xn[R], tn, bn = T(0);  // this block's and the next one's
    T bq[ONE ? 1 : U];
    auto fetch = [&](int k0, T (&x)[R], T &t, T &b) {
        const int k = k0 + lane;
        const bool ok = lane < U && k < kmax;
#pragma unroll
        for (int i = 1; i < R; ++i) x[i] = ql_ld(rD, ok && i < m - k ? k * ldD + ub + i * SZ : -1, 0, T());
        t = ql_ld(rt, ok ? k * SZ : -1, 0, T());
        if (ONE) b = ql_ld(rB, lane < U && k + R < m ? (k + R) * SZ : -1, 0, T());  // the row entering after step k
    };
#pragma unroll
    for (int i = 0; i < R; ++i) w[i] = ql_ld(rB, i < m ? (ONE ? 0 : colb) : -1, i * SZ, T());
    fetch(0, xb, tb, bb);
    if constexpr (!ONE)
        QUnroll<U>::run([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            bq[s] = ql_ld(rB, s + R < m ? colb : -1, (s + R) * SZ, T());
        });
    int k0 = 0;
    T out = T(0);
    auto step = [&](auto sc, auto tc) {
        constexpr int s = decltype(sc)::value;
        constexpr bool TAIL = decltype(tc)::value;
        const int k = k0 + s;
        if (TAIL && k >= kmax) return;
        auto reg = [](int i) { return (i + s) % R; };
        T x[R], p[8];
        p[0] = w[reg(0)];
#pragma unroll
        for (int i = 1; i < 8; ++i) {
            p[i] = T(0);
            if (i < R) {
                x[i] = lane_read(xb[i], s);  // 0 past the last row
                p[i] = x[i] * w[reg(i)];
            }
        }
        const T g0 = (p[3] + p[2]) + (p[1] + p[0]), g1 = (p[7] + p[6]) + (p[5] + p[4]);
        const T v = lane_read(tb, s) * (T(0) + (g1 + g0));
        const T done = w[reg(0)] - v;
#pragma unroll
        for (int i = 1; i < R; ++i) w[reg(i)] = w[reg(i)] - x[i] * v;
        if constexpr (ONE) {
            out = lane == s ? done : out;
            w[reg(0)] = lane_read(bb, s);
        } else {
            ql_st(rB, colb, k * SZ, done);
            w[reg(0)] = bq[s];
            bq[s] = ql_ld(rB, k + U + R < m ? colb : -1, (k + U + R < m ? k + U + R : 0) * SZ, T());
        }
    };
    auto next = [&] {
        if (ONE) ql_st(rB, lane < U && k0 + lane < kmax ? (k0 + lane) * SZ : -1, 0, out);
#pragma unroll
        for (int i = 1; i < R; ++i) xb[i] = xn[i];
        tb = tn;
        bb = bn;
    };
    for (; k0 + U <= kmax; k0 += U) {
        fetch(k0 + U, xn, tn, bn);
        QUnroll<U>::run([&](auto sc) { step(sc, std::false_type{}); });
        next();
    }
    if (k0 < kmax) {
        QUnroll<U>::run([&](auto sc) { step(sc, std::true_type{}); });
        if (ONE) ql_st(rB, lane < U && k0 + lane < kmax ? (k0 + lane) * SZ : -1, 0, out);
    }
    // rows kmax .. kmax+L-1 still in the window
    const int at = kmax % R;
#pragma unroll
    for (int i = 0; i < L; ++i) {
        T z = w[0];
#pragma unroll
        for (int q = 1; q < R; ++q) z = (at + i) % R == q ? w[q] : z;
        ql_st(rB, kmax + i < m && (!ONE || lane == 0) ? (ONE ? 0 : colb) : -1, (kmax + i < m ? kmax + i : 0) * SZ, z);
    }
}

}  // namespace

#define BH_QL_CASES(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7)

int lane_gbqrf_launch(i64 m, i64 n, i64 l, i64 u, BH_QL_T *D, i64 ldd, BH_QL_T *tau, hipStream_t st) {
    using T = BH_QL_T;
    // columns are held from the first row loaded into them (u + l columns) until
    // their last rows have been replaced (l + 1 steps past their own): all in 64 lanes
    if (u + 2 * l > 62 || m >= (1ll << 30) || n >= (1ll << 30) || ldd * n * (i64)sizeof(T) >= (1ll << 31) - (1 << 24) ||
        ldd * (i64)sizeof(T) >= (1ll << 24))
        return -1;
    switch ((int)l) {
#define BH_QL_CASE(Lv)                                                                                         \
    case Lv:                                                                                                   \
        hipLaunchKernelGGL((gbqrf_lane<T, Lv>), dim3(1), dim3(64), 0, st, (int)m, (int)n, (int)u, D, ldd, tau); \
        break;
        BH_QL_CASES(BH_QL_CASE)
#undef BH_QL_CASE
        default:
            return -1;
    }
    BH_LAUNCH_CHECK();
    return BH_OK;
}

int lane_qtb_launch(i64 m, i64 n, i64 l, i64 u, const BH_QL_T *D, i64 ldd, const BH_QL_T *tau, i64 nrhs, BH_QL_T *B,
                    i64 ldb, hipStream_t st) {
    using T = BH_QL_T;
    const i64 lim = (1ll << 31) - (1 << 24);
    if (m >= (1ll << 30) || ldd * n * (i64)sizeof(T) >= lim || ldb * nrhs * (i64)sizeof(T) >= lim) return -1;
    const int kmax = (int)imin(m, n);
    switch ((int)l) {
#define BH_QL_CASE(Lv)                                                                                               \
    case Lv:                                                                                                         \
        if (nrhs == 1)                                                                                               \
            hipLaunchKernelGGL((qtb_lane<T, Lv, true>), dim3(1), dim3(64), 0, st, (int)m, (int)u, D, ldd, n, tau,    \
                               kmax, B, ldb, 1);                                                                     \
        else                                                                                                         \
            hipLaunchKernelGGL((qtb_lane<T, Lv, false>), dim3((unsigned)cdiv(nrhs, 64)), dim3(64), 0, st, (int)m,    \
                               (int)u, D, ldd, n, tau, kmax, B, ldb, (int)nrhs);                                     \
        break;
        BH_QL_CASES(BH_QL_CASE)
#undef BH_QL_CASE
        default:
            return -1;
    }
    BH_LAUNCH_CHECK();
    return BH_OK;
}
#undef BH_QL_CASES
#endif  // BH_QL_T

}  // namespace bh
