// bh_lu_lane.hpp -- narrow-band LU (and fused solve) with one wave per
// system and the subdiagonal count fixed at compile time.
//
// Arithmetic of LAPACK xGBTF2 (LAPACK.gbtrf!, src/banded/BandedLU.jl:98) and
// xGBTRS 'N' (ldiv!, src/banded/linalg.jl:24-30), bit for bit: IDAMAX pivot,
// interchange over the live columns, multipliers a * (1/pivot), updates
// fma(l, -u, a); forward solve fma(l, -b_j, b_i) after the interchange, back
// substitution x_j = b_j / u_jj, fma(u_ij, -x_j, b_i).
//
// Layout: lane c mod 64 holds band column c of the window (columns
// j..j+kl+ku) with its rows j..j+kl in registers; the lane of the retired
// column j takes, when the window reaches it, column j+64.
//
// The kernels are instantiated per element type in bh_lu_lane_d.hip and
// bh_lu_lane_s.hip (define BH_LANE_T before including this header); other
// files see only the descriptor and the launchers.
#pragma once
#include "bh_common.hpp"
#include "bh_cut.hpp"

#include <type_traits>

namespace bh {

// One system of a batch, in schedule order.
struct BatchDesc {
    i64 ab_off;   // element offset of the system's padded AB
    i64 vec_off;  // element offset of its b / ipiv
    int n, kl, ku, cls, sys;
};

// Single-system gbtrf through the rotating-register kernel (kl <= 16, kl + ku <= 63, band storage under 2 GiB), or -1.  With a cut it
// runs the blocks of a cut system, one wave each; with cut->g.p == 0 it does
// nothing unless cut->flags say that the gate is closed.
int lane_gbtrf_launch(i64 m, i64 n, i64 kl, i64 ku, double *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                      const LuCut<double> *cut);
int lane_gbtrf_launch(i64 m, i64 n, i64 kl, i64 ku, float *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                      const LuCut<float> *cut);
// its widths 9 .. 15, compiled in units of their own (bh_lu_lane_wide_{d,s}.hip)
int lane_gbtrf_launch_wide(i64 m, i64 n, i64 kl, i64 ku, double *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                           const LuCut<double> *cut);
int lane_gbtrf_launch_wide(i64 m, i64 n, i64 kl, i64 ku, float *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                           const LuCut<float> *cut);
// The persistent batched gbsv kernel over a schedule of nsys descriptors.
int lane_batch_launch(unsigned blocks, unsigned threads, hipStream_t st, const BatchDesc *desc, int nsys, double *AB,
                      double *B, i64 *ipiv, i64 *info);
int lane_batch_launch(unsigned blocks, unsigned threads, hipStream_t st, const BatchDesc *desc, int nsys, float *AB,
                      float *B, i64 *ipiv, i64 *info);

#ifdef BH_LANE_T
namespace {

template <int K>
struct SK {
    static constexpr int value = K;
};
template <int N>
struct SUnroll {
    template <class F>
    __device__ __forceinline__ static void run(F &&f) {
        SUnroll<N - 1>::run(f);
        f(SK<N - 1>{});
    }
};
template <>
struct SUnroll<0> {
    template <class F>
    __device__ __forceinline__ static void run(F &&) {}
};

__device__ __forceinline__ int smin(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ int smax(int a, int b) { return a > b ? a : b; }

// ---------------------------------------------------------------- rotating-register form
// The same arithmetic as small_gbsv_wave, restructured so that a step is a
// short straight-line sequence:
//  * KL (the subdiagonal count) is a compile-time constant and the window
//    has exactly R = KL + 1 rows; the steps are unrolled in blocks of U (a
//    multiple of R), and row i of step s lives in register (i + s) mod R, so
//    rows never move between registers;
//  * pivot: every lane finds the first largest |a| of its own column (a NaN is
//    never larger, and never beaten in row 0: the reference IDAMAX choice);
//    the row and value of the owner become uniform with one readlane each;
//  * multipliers: every lane scales its own column by the uniform reciprocal,
//    the owner's are read into scalar registers, which the updates take as
//    operands, and stored from the owner's lane;
//  * addresses: a step's uniform part is the instruction's scalar offset, a
//    lane's part one 24-bit product;
//  * memory goes through buffer resources: a lane with nothing to load or
//    store passes an offset past the end (the hardware returns 0 / drops the
//    store), so no access sits in a branch and the memory counter waits stay
//    exact; the incoming row of each step is loaded U steps ahead.
// What bounds a step is the issue of one wave's instructions (about 6.4 cycles
// each, measured over both forms of the step): n = 10000, (4,4), FP64 with
// interchanges, 510 -> 385 ns a step when the multipliers left the LDS
// permutes, the scalar compares and the 64-bit address products.
constexpr int kBufWord3 = 0x00020000;  // word 3 of a raw buffer resource (gfx9 family)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *p, i64 bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, kBufWord3);
}
// off: the lane's byte offset (past the end: nothing moves), uni: a uniform one
__device__ __forceinline__ double buf_ld(__amdgpu_buffer_rsrc_t r, int off, double, int uni = 0) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, uni, 0));
}
__device__ __forceinline__ float buf_ld(__amdgpu_buffer_rsrc_t r, int off, float, int uni = 0) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, uni, 0));
}
__device__ __forceinline__ void buf_st(__amdgpu_buffer_rsrc_t r, int off, double v, int uni = 0) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, off, uni, 0);
}
__device__ __forceinline__ void buf_st(__amdgpu_buffer_rsrc_t r, int off, float v, int uni = 0) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, uni, 0);
}
__device__ __forceinline__ void buf_st64(__amdgpu_buffer_rsrc_t r, int off, long long v) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, off, 0, 0);
}
// whether a uniform value is not +-0, in scalar integer arithmetic
__device__ __forceinline__ bool nonzero_bits(double x) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    return (((unsigned)(b >> 32) & 0x7fffffffu) | (unsigned)b) != 0;
}
__device__ __forceinline__ bool nonzero_bits(float x) { return (__builtin_bit_cast(unsigned, x) & 0x7fffffffu) != 0; }
template <typename T, int KL, bool SOLVE, int UMIN>
__device__ __forceinline__ int lane_gbsv_wave(int m, int n, int ku, T *__restrict__ ab, i64 ld, i64 *__restrict__ ipiv,
                              T *__restrict__ b) {
    constexpr int R = KL + 1;
    constexpr int U = R * ((UMIN - 1 + R) / R);  // steps per unrolled block (>= UMIN, a multiple of R)
    constexpr int SZ = (int)sizeof(T);
    const int lane = (int)__lane_id();
    const int kv = KL + ku;
    const int mn = smin(m, n);
    if (mn == 0) return 0;
    const __amdgpu_buffer_rsrc_t rab = buf_rsrc(ab, ld * (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rip = buf_rsrc(ipiv, (i64)mn * 8);
    const __amdgpu_buffer_rsrc_t rb = buf_rsrc(b, SOLVE ? (i64)n * SZ : 0);
    // byte offset of A(r, c) in AB, or -1 (past the end) when it is not stored there
    auto off_a = [&](int r, int c) -> int {
        const bool ok = r >= 0 && r < m && c >= 0 && c < n && c - r <= ku && r - c <= KL;
        return ok ? (int)(((i64)c * ld + kv + r - c) * SZ) : -1;
    };
    // the row entering at the end of step j: row j+1+KL of the lane's column then
    auto off_in = [&](int j) -> int {
        const int c = (j + 1) + ((lane - (j + 1)) & 63);
        return j < mn ? off_a(j + 1 + KL, c) : -1;
    };
    auto off_bin = [&](int j) -> int {
        const int e = j + 1 + KL;
        return (SOLVE && j < mn && e < n) ? e * SZ : -1;
    };

    T y[R], pre[U];
    T bw[R], bpre[U];
#pragma unroll
    for (int i = 0; i < R; ++i) y[i] = buf_ld(rab, off_a(i, lane), T());
    SUnroll<U>::run([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        pre[s] = buf_ld(rab, off_in(s), T());
    });
    if (SOLVE) {
#pragma unroll
        for (int i = 0; i < R; ++i) bw[i] = buf_ld(rb, i < n ? i * SZ : -1, T());
        SUnroll<U>::run([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            bpre[s] = buf_ld(rb, off_bin(s), T());
        });
    }
    // Strides of a step's addresses: with d = (lane - j) mod 64 the lane's
    // column is j + d, and row j of it lies (j*ld + kv) + d*(ld - 1) elements
    // into AB: a uniform part (the instruction's scalar offset) and one
    // 24-bit product.
    const int dstep = (int)(ld - 1) * SZ, ldb = (int)ld * SZ, kvb = kv * SZ;
    const int lane0 = lane == 0 ? 0 : -1;  // stores of one uniform value
    // A lane takes column j+64 when column j retires; rows of column j it still
    // holds when j+64 enters the window must read as zero.  Outside the
    // window a lane's rows never move, so one is replaced by an incoming row
    // per step, all of them before j+64 enters unless 2*KL + ku > 63.
    const bool clear_retired = 2 * KL + ku > 63;
    int ju = 0, info = 0, j0 = 0;
    int ip = 0;  // pivots of the current U steps, step s in lane s

    auto step = [&](auto sc, auto tc) {
        constexpr int s = decltype(sc)::value;
        constexpr bool TAIL = decltype(tc)::value;
        const int j = j0 + s;
        if (TAIL && j >= mn) return;
        const int own = j & 63;
        const int km = TAIL ? smin(KL, m - 1 - j) : KL;
        auto reg = [](int i) { return (i + s) % R; };
        // pivot: the first row of the largest |a|, found by every lane for its
        // own column (a NaN is never larger, and never beaten in row 0); the
        // owner's row and value become uniform
        T bv = y[reg(0)];
        int jpl = 0;
#pragma unroll
        for (int i = 1; i < R; ++i) {
            const bool gt = dabs(y[reg(i)]) > dabs(bv);
            if (!TAIL || i <= km) {
                bv = gt ? y[reg(i)] : bv;
                jpl = gt ? i : jpl;
            }
        }
        const int jp = __builtin_amdgcn_readlane(jpl, own);
        const T pv = lane_read(bv, own);
        const bool nz = nonzero_bits(pv);  // NaN counts as nonzero, as in LAPACK's test
        const int juj = smin(j + jp + ku, n - 1);
        ju = nz && juj > ju ? juj : ju;
        info = !nz && info == 0 ? j + 1 : info;
        // interchange rows 0 and jp over columns j..ju only: a lane outside
        // them keeps its rows in place, so the rows a retired column leaves
        // behind are overwritten by incoming rows within R steps.  (Selects on
        // scalar conditions: a chain of branches costs copies of every row
        // where they join.)
        const int d = (lane - j) & 63;
        if (jp != 0) {
            const bool live = d <= ju - j;
            const T t0 = y[reg(0)], b0 = SOLVE ? bw[reg(0)] : T(0);
            T t = t0, b1 = b0;
#pragma unroll
            for (int i = 1; i < R; ++i) {
                const bool sw = (jp == i) & live;
                t = sw ? y[reg(i)] : t;
                y[reg(i)] = sw ? t0 : y[reg(i)];
                if (SOLVE) {
                    b1 = jp == i ? bw[reg(i)] : b1;
                    bw[reg(i)] = jp == i ? b0 : bw[reg(i)];
                }
            }
            y[reg(0)] = t;
            if (SOLVE) bw[reg(0)] = b1;
        }
        // multipliers: every lane scales its own column; lane own's are read
        // into scalar registers, which the updates take as operands
        const T rcp = nz ? T(1) / pv : T(1);
        T lc[R], l[R];
#pragma unroll
        for (int i = 1; i < R; ++i) {
            lc[i] = y[reg(i)] * rcp;
            l[i] = lane_read(lc[i], own);
        }
        // U row j (lanes of columns j..j+kv; the pivot from lane own), then
        // column j's multipliers from lane own
        const int rowb = j * ldb + kvb;
        buf_st(rab, d <= smin(kv, n - 1 - j) ? (int)__umul24(d, dstep) : -1, y[reg(0)], rowb);
        const int vown = d == 0 ? 0 : -(1 << 30);
#pragma unroll
        for (int i = 1; i < R; ++i)
            if (!TAIL || i <= km) buf_st(rab, vown + i * SZ, lc[i], rowb);
        ip = lane == s ? j + jp + 1 : ip;
        // rank-1 update of columns j+1..ju, rows 1..km (a zero pivot updates nothing)
        if ((unsigned)(d - 1) < (unsigned)(nz ? ju - j : 0)) {
            const T nu = -y[reg(0)];
#pragma unroll
            for (int i = 1; i < R; ++i)
                if (!TAIL || i <= km) y[reg(i)] = dfma(l[i], nu, y[reg(i)]);
        }
        if (SOLVE) {
            // forward substitution step j (xGBTRS: interchange, then the L column)
            const T nb = -bw[reg(0)];
            const int kb = TAIL ? smin(KL, n - 1 - j) : KL;
#pragma unroll
            for (int i = 1; i < R; ++i)
                if (!TAIL || i <= kb) bw[reg(i)] = dfma(l[i], nb, bw[reg(i)]);
            buf_st(rb, lane0, bw[reg(0)], j * SZ);
            bw[reg(0)] = bpre[s];
            bpre[s] = buf_ld(rb, off_bin(j + U), T());
        }
        if (clear_retired && d == 0) {
#pragma unroll
            for (int i = 1; i < R; ++i) y[reg(i)] = T(0);
        }
        y[reg(0)] = pre[s];
        {
            const int J = j + U + 1, dj = (lane - J) & 63;  // the row entering at the end of step j+U
            const int lim = (J <= mn && J + KL < m) ? smin(kv, n - 1 - J) : -1;
            pre[s] = buf_ld(rab, dj <= lim ? (int)__umul24(dj, dstep) : -1, T(), J * ldb + kvb + KL * SZ);
        }
    };
    auto put_pivots = [&] {
        buf_st64(rip, (lane < U && j0 + lane < mn) ? (j0 + lane) * 8 : -1, (long long)ip);
    };
    const int jmain = smin(mn, m - KL);  // steps before it have km == KL
    for (; j0 + U <= jmain; j0 += U) {
        SUnroll<U>::run([&](auto sc) { step(sc, std::false_type{}); });
        put_pivots();
    }
    for (; j0 < mn; j0 += U) {
        SUnroll<U>::run([&](auto sc) { step(sc, std::true_type{}); });
        put_pivots();
    }

    // Fill-in rows LAPACK zeroes that no U row covered (rows >= m).
    {
        const int c_lo = smax(ku + 1, m + ku), c_hi = smin(n, mn + kv);
        for (int c = c_lo + lane; c < c_hi; c += 64) {
            for (int q = smax(0, kv - c); q < KL; ++q)
                if (c - kv + q >= m) ab[(i64)c * ld + q] = T(0);
        }
    }
    if (SOLVE) {
        // back substitution: lane t holds b_{j-t}, t = 0 .. kl+ku
        T w = buf_ld(rb, (lane <= kv && n - 1 - lane >= 0) ? (n - 1 - lane) * SZ : -1, T());
        T ur[U], br[U];
        auto off_u = [&](int j) { return (j >= 0 && lane <= smin(kv, j)) ? (int)(((i64)j * ld + kv - lane) * SZ) : -1; };
        auto off_br = [&](int j) { return (j >= 0 && j - 1 - kv >= 0) ? (j - 1 - kv) * SZ : -1; };
        SUnroll<U>::run([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            ur[s] = buf_ld(rab, off_u(n - 1 - s), T());
            br[s] = buf_ld(rb, off_br(n - 1 - s), T());
        });
        for (int jb = n - 1; jb >= 0; jb -= U) {
            SUnroll<U>::run([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                const int j = jb - s;
                if (j >= 0) {
                    const T xj = lane_read(w, 0) / lane_read(ur[s], 0);
                    buf_st(rb, lane == 0 ? j * SZ : -1, xj);
                    if (lane >= 1 && lane <= smin(kv, j)) w = dfma(ur[s], -xj, w);
                    w = wave_down1(w, T(0));
                    if (lane == kv) w = br[s];
                    ur[s] = buf_ld(rab, off_u(j - U), T());
                    br[s] = buf_ld(rb, off_br(j - U), T());
                }
            });
        }
    }
    return info;
}

template <typename T, int KL>
__global__ void __launch_bounds__(64) gbtrf_lane_kernel(int m, int n, int ku, T *ab, i64 ld, i64 *ipiv, i64 *info,
                                                        LuCut<T> cut) {
    if (cut.g.p > 0) {  // this wave's block of a cut system
        if (cut_closed(cut.flags)) return;
        const int blk = blockIdx.x;
        ab = cut.block_ab(blk);
        ld = cut.H;
        m = cut.rows(blk);
        n = cut.cols(blk);
        ipiv = cut.ipiv + (i64)blk * cut.g.span();
        info = cut.info + 2 * blk;
    } else if (cut.flags && !cut_failed(cut.flags)) {
        return;  // the gate is open: the blocks of a cut system do it
    }
    const int r = lane_gbsv_wave<T, KL, false, 16>(m, n, ku, ab, ld, ipiv, nullptr);
    if (threadIdx.x == 0) *info = r;
}


// One body per subdiagonal count (inlined; the kernel's register budget is
// that of the widest).
// One outlined body per subdiagonal count, so the batched kernel is a switch
// over calls rather than nine inlined copies.
template <typename T, int KL>
__device__ __noinline__ int batch_sys(int n, int ku, T *ab, i64 ld, i64 *ip, T *b) {
    return lane_gbsv_wave<T, KL, true, 8>(n, n, ku, ab, ld, ip, b);
}

template <typename T>
__device__ __forceinline__ int batch_one(const BatchDesc &d, T *AB, T *Bv, i64 *IP) {
    const i64 ld = 2 * d.kl + d.ku + 1;
    T *ab = AB + d.ab_off;
    T *b = Bv + d.vec_off;
    i64 *ip = IP + d.vec_off;
    switch (d.kl) {
#define BH_BATCH_CASE(KLv) \
    case KLv:              \
        return batch_sys<T, KLv>(d.n, d.ku, ab, ld, ip, b);
        BH_BATCH_CASE(0)
        BH_BATCH_CASE(1)
        BH_BATCH_CASE(2)
        BH_BATCH_CASE(3)
        BH_BATCH_CASE(4)
        BH_BATCH_CASE(5)
        BH_BATCH_CASE(6)
        BH_BATCH_CASE(7)
        default:
            return batch_sys<T, 8>(d.n, d.ku, ab, ld, ip, b);
#undef BH_BATCH_CASE
    }
}

// Persistent: wave w of the W resident waves solves systems w, w + W,
// w + 2W, ... of the schedule (the plan orders the systems so that this
// visit order balances the work).  All loop bounds are wave-uniform
// (readfirstlane), so the step loops stay scalar loops.
template <typename T>
__global__ void __launch_bounds__(256) gbsv_batched_kernel(const BatchDesc *__restrict__ desc, int nsys, T *AB,
                                                           T *Bv, i64 *IP, i64 *info) {
    auto uni64 = [](i64 v) {
        const int lo = __builtin_amdgcn_readfirstlane((int)(v & 0xffffffff));
        const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
        return (i64)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
    };
    const int nw = (int)(gridDim.x * (blockDim.x >> 6));
    const int w0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
    for (int q = w0; q < nsys; q += nw) {
        const BatchDesc dv = desc[q];
        BatchDesc d;
        d.ab_off = uni64(dv.ab_off);
        d.vec_off = uni64(dv.vec_off);
        d.n = __builtin_amdgcn_readfirstlane(dv.n);
        d.kl = __builtin_amdgcn_readfirstlane(dv.kl);
        d.ku = __builtin_amdgcn_readfirstlane(dv.ku);
        d.cls = __builtin_amdgcn_readfirstlane(dv.cls);
        d.sys = __builtin_amdgcn_readfirstlane(dv.sys);
        const int r = batch_one<T>(d, AB, Bv, IP);
        if (d.sys >= 0 && __lane_id() == 0) info[d.sys] = r;
    }
}

}  // namespace

#ifdef BH_LANE_WIDE
int lane_gbtrf_launch_wide(i64 m, i64 n, i64 kl, i64 ku, BH_LANE_T *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                      const LuCut<BH_LANE_T> *cut) {
    using T = BH_LANE_T;
    const i64 nb = cut && cut->g.p > 0 ? cut->g.span() : n;  // a block's copy holds span() columns
    if (kl + ku > 63 || m >= (1ll << 30) || n >= (1ll << 30) || ldab * nb * (i64)sizeof(T) >= (1ll << 31) ||
        ldab * (i64)sizeof(T) >= (1ll << 24))
        return -1;
    const int mi = (int)m, ni = (int)n, ui = (int)ku;
    const LuCut<T> c = cut ? *cut : LuCut<T>{};
    const dim3 grid(c.g.p > 0 ? (unsigned)c.g.p : 1u);
    switch ((int)kl) {
#define BH_LANE_CASE(KLv)                                                                                       \
    case KLv:                                                                                                   \
        hipLaunchKernelGGL((gbtrf_lane_kernel<T, KLv>), grid, dim3(64), 0, st, mi, ni, ui, ab, ldab, ipiv,      \
                           dinfo, c);                                                                           \
        break;
        BH_LANE_CASE(9) BH_LANE_CASE(10) BH_LANE_CASE(11) BH_LANE_CASE(12) BH_LANE_CASE(13) BH_LANE_CASE(14)
        BH_LANE_CASE(15)
#undef BH_LANE_CASE
        default:
            return -1;
    }
    BH_LAUNCH_CHECK();
    return BH_OK;
}

#else
int lane_gbtrf_launch(i64 m, i64 n, i64 kl, i64 ku, BH_LANE_T *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                      const LuCut<BH_LANE_T> *cut) {
    using T = BH_LANE_T;
    const i64 nb = cut && cut->g.p > 0 ? cut->g.span() : n;  // a block's copy holds span() columns
    if (kl + ku > 63 || m >= (1ll << 30) || n >= (1ll << 30) || ldab * nb * (i64)sizeof(T) >= (1ll << 31) ||
        ldab * (i64)sizeof(T) >= (1ll << 24))
        return -1;
    const int mi = (int)m, ni = (int)n, ui = (int)ku;
    const LuCut<T> c = cut ? *cut : LuCut<T>{};
    const dim3 grid(c.g.p > 0 ? (unsigned)c.g.p : 1u);
    switch ((int)kl) {
#define BH_LANE_CASE(KLv)                                                                                       \
    case KLv:                                                                                                   \
        hipLaunchKernelGGL((gbtrf_lane_kernel<T, KLv>), grid, dim3(64), 0, st, mi, ni, ui, ab, ldab, ipiv,      \
                           dinfo, c);                                                                           \
        break;
        BH_LANE_CASE(0) BH_LANE_CASE(1) BH_LANE_CASE(2) BH_LANE_CASE(3) BH_LANE_CASE(4)
        BH_LANE_CASE(5) BH_LANE_CASE(6) BH_LANE_CASE(7) BH_LANE_CASE(8) BH_LANE_CASE(16)
#undef BH_LANE_CASE
        default:
            return kl <= 15 ? lane_gbtrf_launch_wide(m, n, kl, ku, ab, ldab, ipiv, dinfo, st, cut) : -1;
    }
    BH_LAUNCH_CHECK();
    return BH_OK;
}

int lane_batch_launch(unsigned blocks, unsigned threads, hipStream_t st, const BatchDesc *desc, int nsys,
                      BH_LANE_T *AB, BH_LANE_T *B, i64 *ipiv, i64 *info) {
    hipLaunchKernelGGL(gbsv_batched_kernel<BH_LANE_T>, dim3(blocks), dim3(threads), 0, st, desc, nsys, AB, B, ipiv,
                       info);
    BH_LAUNCH_CHECK();
    return BH_OK;
}
#endif  // BH_LANE_WIDE
#endif  // BH_LANE_T

}  // namespace bh
