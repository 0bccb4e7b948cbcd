// bh_gbtrf.hip -- partial-pivot band LU on gfx950.
//
// Restates LAPACK xGBTF2, the routine the reference's LAPACK.gbtrf!
// (src/banded/BandedLU.jl:98) runs for ku <= 64, step for step:
//   for each column j: zero the fill-in rows of column j+kv; pick the pivot
//   as the first row of max |a| among rows j..j+km (IDAMAX); record ipiv;
//   swap rows across columns j..ju; scale the multipliers by the rounded
//   reciprocal of the pivot; rank-1 update a_ic = fma(l_i, -u_jc, a_ic).
// The rounding of every step matches the CPU routine, so factors and pivots
// are bit-identical to it.
//
// Kernel: one workgroup runs the column chain of one system; the working
// window lives in global memory (L2-resident: at most (2kl+ku+1) x (kl+ku+1)
// entries are live) and the phases of a step are separated by workgroup
// barriers.  Each phase is spread over the workgroup's lanes.
#include "bh_common.hpp"
#include "bh_cut.hpp"
#include "bh_lu_lane.hpp"

#include <cstdlib>
#include <cstring>

namespace bh {

constexpr int kLuThreads = 256;

template <typename T>
struct LuSys {
    T *ab;
    i64 *ipiv;
    i64 m, n, kl, ku, ldab;
};

// Argmax over |col[kv+t]|, t in [0, km], first index on ties; whole block.
template <typename T>
__device__ __forceinline__ i64 block_pivot(const T *col, i64 km, T *sval, int *sidx) {
    T best = T(-1);
    int bidx = 0x7fffffff;
    for (i64 t = threadIdx.x; t <= km; t += blockDim.x) {
        T v = dabs(col[t]);
        if (v > best) {  // strictly greater keeps the first index per thread
            best = v;
            bidx = (int)t;
        }
    }
    // wave reduction: larger value wins, equal values keep the smaller index
    for (int off = 32; off > 0; off >>= 1) {
        T ov = __shfl_xor(best, off, 64);
        int oi = __shfl_xor(bidx, off, 64);
        if (ov > best || (ov == best && oi < bidx)) {
            best = ov;
            bidx = oi;
        }
    }
    const int wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sval[wid] = best;
        sidx[wid] = bidx;
    }
    __syncthreads();
    T b = sval[0];
    int bi = sidx[0];
    for (int w = 1; w < nw; ++w) {
        if (sval[w] > b || (sval[w] == b && sidx[w] < bi)) {
            b = sval[w];
            bi = sidx[w];
        }
    }
    __syncthreads();
    return bi == 0x7fffffff ? 0 : bi;
}

template <typename T>
__device__ void gbtf2_block(const LuSys<T> s, i64 *info_out) {
    __shared__ T sval[16];
    __shared__ int sidx[16];
    const i64 kl = s.kl, ku = s.ku, kv = kl + ku, ld = s.ldab, m = s.m, n = s.n;
    T *ab = s.ab;
    i64 info = 0;
    if (m == 0 || n == 0) {
        if (threadIdx.x == 0 && info_out) *info_out = 0;
        return;
    }
    // fill-in rows of columns ku+1 .. min(kv,n)-1 start at zero
    for (i64 c = ku + 1; c < imin(kv, n); ++c)
        for (i64 r = kv - c + threadIdx.x; r < kl; r += blockDim.x) ab[c * ld + r] = T(0);
    __syncthreads();
    i64 ju = 0;
    const i64 steps = imin(m, n);
    for (i64 j = 0; j < steps; ++j) {
        if (j + kv < n)
            for (i64 r = threadIdx.x; r < kl; r += blockDim.x) ab[(j + kv) * ld + r] = T(0);
        const i64 km = imin(kl, m - 1 - j);
        T *colj = ab + j * ld + kv;  // colj[t] = A(j+t, j)
        const i64 jp = block_pivot(colj, km, sval, sidx);
        if (threadIdx.x == 0) s.ipiv[j] = jp + j + 1;
        const T piv = colj[jp];
        if (piv != T(0)) {
            ju = imax(ju, imin(j + ku + jp, n - 1));
            if (jp != 0) {
                for (i64 c = j + threadIdx.x; c <= ju; c += blockDim.x) {
                    T *p = ab + c * ld + kv + jp + j - c;
                    T *q = ab + c * ld + kv + j - c;
                    T tmp = *p;
                    *p = *q;
                    *q = tmp;
                }
                __syncthreads();
            }
            if (km > 0) {
                const T r = T(1) / colj[0];
                for (i64 t = 1 + threadIdx.x; t <= km; t += blockDim.x) colj[t] = colj[t] * r;
                __syncthreads();
                const i64 ncol = ju - j;
                const i64 tot = km * ncol;
                for (i64 e = threadIdx.x; e < tot; e += blockDim.x) {
                    const i64 cc = e / km, t = e - cc * km + 1, c = j + 1 + cc;
                    T *colc = ab + c * ld;
                    const T negu = -colc[kv + j - c];
                    colc[kv + j + t - c] = dfma(colj[t], negu, colc[kv + j + t - c]);
                }
            }
        } else if (info == 0) {
            info = j + 1;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0 && info_out) *info_out = info;
}

template <typename T>
__global__ void __launch_bounds__(kLuThreads) gbtf2_single(LuSys<T> s, i64 *info_out) {
    gbtf2_block<T>(s, info_out);
}

template <typename T>
int reg_gbtrf_launch(i64 m, i64 n, i64 kl, i64 ku, T *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st);
template <typename T>
int blk_gbtrf_launch(i64 m, i64 n, i64 kl, i64 ku, T *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                     const LuCut<T> *cut);
template <typename T>
int small_gbtrf_launch(i64 m, i64 n, i64 kl, i64 ku, T *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st);
template <typename T>
int mfma_gbtrf_launch(i64 m, i64 n, i64 kl, i64 ku, T *ab, i64 ldab, i64 *ipiv, i64 *dinfo, hipStream_t st,
                      const LuCut<T> *cut);

// Kernel choice: BANDEDHIP_LU_KERNEL = "small" | "blk" | "reg" | "global" |
// "mfma" forces one (where it applies).  By default, as LAPACK xGBTRF
// decides between its unblocked and blocked code (ILAENV block size 32 for
// ku > 64, blocked when the block size is at most kl): the MFMA-blocked
// kernel for ku >= 65 and kl >= 32, whose pivots are xGBTRF's and whose
// factors agree with it to rounding.  Otherwise the xGBTF2-exact kernels:
// the one-wave kernel for kl <= 16, the register-window blocked kernel for
// kl >= 16 where that did not apply, the per-step register kernel otherwise.
constexpr i64 kLongLu = 16384;  // systems at least this long take the MFMA factorisation (kl, ku >= 8)

static int lu_kernel_override() {
    const char *e = getenv("BANDEDHIP_LU_KERNEL");
    if (!e) return 0;
    if (!strcmp(e, "blk")) return 1;
    if (!strcmp(e, "reg")) return 2;
    if (!strcmp(e, "global")) return 3;
    if (!strcmp(e, "small")) return 4;
    if (!strcmp(e, "mfma")) return 5;
    return 0;
}

// ---------------------------------------------------------------- cut systems
// (bh_cut.hpp).  The seams are checked on the multipliers and pivots alone:
// at step t = c - (kl+ku) the rows still active hold nothing in columns >= c
// yet (the rows read so far end before it), so two runs whose multipliers
// and pivots agree over columns t .. c-1 do the same operations on the same
// entries of every column from c on.

// Copies of the blocks' columns, fill-in rows zeroed as LAPACK zeroes them
// (slots outside the matrix keep what the caller has there).
template <typename T>
__global__ void __launch_bounds__(256) lu_cut_copy(LuCut<T> cut, const T *__restrict__ ab, i64 ld, int kv) {
    if (cut_closed(cut.flags)) return;
    const int blk = blockIdx.y, H = cut.H, s0 = cut.g.start(blk);
    const int tot = cut.cols(blk) * H;
    T *dst = cut.block_ab(blk);
    for (int e = blockIdx.x * 256 + threadIdx.x; e < tot; e += gridDim.x * 256) {
        const int c = e / H, r = e - c * H;
        const bool fill = r < cut.kl && s0 + c + r - kv >= 0;
        dst[e] = fill ? T(0) : ab[(i64)(s0 + c) * ld + r];
    }
    if (blockIdx.x == 0 && threadIdx.x < 2) cut.info[2 * blk + threadIdx.x] = 0;
}

// Block i against block i-1 over the `cmp` columns before its own begin.
template <typename T>
__global__ void __launch_bounds__(256) lu_cut_check(LuCut<T> cut, int kv, int cmp, int *flags) {
    if (cut_closed(flags)) return;
    const int blk = blockIdx.x, H = cut.H;
    bool bad = threadIdx.x < 2 && cut.info[2 * blk + threadIdx.x] != 0;
    if (cut.g.start(blk) > 0) {
        const int c0 = cut.g.own(blk) - cmp, a0 = c0 - cut.g.start(blk - 1), b0 = c0 - cut.g.start(blk);
        const T *a = cut.block_ab(blk - 1), *b = cut.block_ab(blk);
        // a wave to a column, four columns in flight
#pragma unroll 4
        for (int c = threadIdx.x >> 6; c < cmp; c += 4)
            for (int r = kv + 1 + (threadIdx.x & 63); r <= kv + cut.kl; r += 64)
                bad |= cut_differ(a[(i64)(a0 + c) * H + r], b[(i64)(b0 + c) * H + r]);
        const i64 *pa = cut.ipiv + (i64)(blk - 1) * cut.g.span(), *pb = cut.ipiv + (i64)blk * cut.g.span();
        for (int c = threadIdx.x; c < cmp; c += 256) bad |= pa[a0 + c] - a0 != pb[b0 + c] - b0;
    }
    if (__syncthreads_or(bad) && threadIdx.x == 0) atomicOr(flags + 1, 1);
}

template <typename T>
__global__ void __launch_bounds__(256) lu_cut_commit(LuCut<T> cut, T *__restrict__ ab, i64 ld, i64 *__restrict__ ipiv,
                                                     int *host) {
    const bool failed = cut_failed(cut.flags);
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) cut_tell(host, failed);
    if (failed) return;
    const int blk = blockIdx.y, H = cut.H, s0 = cut.g.start(blk), c0 = cut.g.own(blk), nc = cut.g.end(blk) - c0;
    const T *src = cut.block_ab(blk) + (i64)(c0 - s0) * H;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < nc * H; e += gridDim.x * 256) {
        const int c = e / H, r = e - c * H;
        ab[(i64)(c0 + c) * ld + r] = src[e];
    }
    const i64 *pv = cut.ipiv + (i64)blk * cut.g.span() + (c0 - s0);
    for (int c = blockIdx.x * 256 + threadIdx.x; c < nc; c += gridDim.x * 256) ipiv[c0 + c] = pv[c] + s0;
}

static i64 up16(i64 x) { return (x + 15) & ~(i64)15; }

// Blocks for n columns: W steps of lead-in, own steps so that `blocks` of
// them fill the chip.  Measured over whole systems (n = 65536 and 262144,
// bands from (1,1) to (128,128), N(0,1) + 2(kl+ku) I and U[0,1) + (kl+ku+1) I,
// k = max(kl, ku)): every seam agrees from 8 k (FP32) and from 12 k (FP64) on
// where kl = ku, earlier where they differ; 10 and 16 at k = 4.  A longer
// lead-in costs little (FP64 (128,128): 3.15 ms at 12 k, 3.76 at 16 k, 58 ms
// when it is too short), so some is added; `tries` times four.
template <typename T>
static CutGeom lu_cut_geom(i64 n, i64 kl, i64 ku, i64 blocks, int tries) {
    const i64 k = imax(kl, ku);
    i64 W = up16(imax(sizeof(T) == 8 ? 14 * k + 64 : 9 * k + 64, up16(kl + ku) + 16));
    for (int t = 0; t < tries; ++t) W *= 4;
    const i64 L = imax(64, up16(cdiv(n, blocks)));
    CutGeom g{(int)n, (int)L, (int)W, (int)cdiv(n, L)};
    // a block's L + W steps must be well under the chain's n
    if (n >= (1ll << 29) || 3 * (L + W) > n) g.p = 0;
    return g;
}

// Factor a square system by blocks.  Tried for sampled columns that exceed
// 1.25 times the rest of their column: the measured families are at 2 and
// more, and a matrix near 1 (the second difference) forgets too slowly for
// its bits to agree, so it would only pay.  Measured, whole gbtrf call against the
// sequential kernels: FP64 (8,8) n = 10000 0.17 ms against 5.3, (16,16)
// n = 262144 0.75 against 125, (128,128) n = 65536 2.7 against 57.6 (FP32 1.29
// against 37); what bounds it is the L + W steps of one block.  The host learns
// the gate's word while the sequential kernel, launched behind it, begins (or
// finds the gate open and ends): a matrix that is not dominant pays the gate, not
// the blocks' launches too.  kCutDone: the factors and pivots are in place,
// info 0; kCutLaunched: the sequential kernel runs already; kCutNot: neither.
int blk_shape_for(i64 kl, i64 ku);
size_t mfma_lds_bytes(i64 kl, i64 elem);

enum LuKernel { kLuNone, kLuMfma, kLuLane, kLuBlk };

template <typename T>
static int lu_kernel_launch(LuKernel kind, i64 n, i64 kl, i64 ku, T *ab, i64 ldab, i64 *ipiv, i64 *dinfo,
                            hipStream_t st, const LuCut<T> *cut) {
    switch (kind) {
        case kLuMfma: return mfma_gbtrf_launch<T>(n, n, kl, ku, ab, ldab, ipiv, dinfo, st, cut);
        case kLuLane: return lane_gbtrf_launch(n, n, kl, ku, ab, ldab, ipiv, dinfo, st, cut);
        case kLuBlk: return blk_gbtrf_launch<T>(n, n, kl, ku, ab, ldab, ipiv, dinfo, st, cut);
        default: return -1;
    }
}

enum CutOutcome { kCutNot, kCutLaunched, kCutDone };

template <typename T>
static int gbtrf_cut(LuKernel kind, i64 n, i64 kl, i64 ku, T *ab, i64 ldab, i64 *ipiv, i64 *dinfo, CutOutcome *out) {
    *out = kCutNot;
    if (kl < 1 || !cut_enabled()) return BH_OK;
    hipStream_t st = stream();
    const int kv = (int)(kl + ku), H = (int)(2 * kl + ku + 1);
    // one workgroup per CU for the MFMA and the blocked kernel (their LDS), one wave per SIMD for the lane kernel
    const i64 blocks = kind == kLuLane ? 1024 : 256;
    struct Free {
        void *p = nullptr;
        hipStream_t st;
        ~Free() { cut_free(p, st); }
    };
    for (int tries = 0; tries < 2; ++tries) {
        const CutGeom g = lu_cut_geom<T>(n, kl, ku, blocks, tries);
        int *host = g.p > 0 ? cut_host_words() : nullptr;
        if (!host) return BH_OK;
        const size_t ba = (((size_t)g.p * g.span() * H * sizeof(T)) + 255) & ~(size_t)255;
        const size_t bp = (size_t)g.p * g.span() * sizeof(i64), bi = (size_t)g.p * 2 * sizeof(i64);
        Free mem;
        mem.st = st;
        char *ws = (char *)(mem.p = cut_alloc(ba + bp + bi + 256, st));
        if (!ws) return BH_OK;
        int *flags = (int *)(ws + ba + bp + bi);
        const LuCut<T> cut{g, flags, (T *)ws, (i64 *)(ws + ba), (i64 *)(ws + ba + bp), H, (int)kl};
        hipLaunchKernelGGL(cut_gate<T>, dim3(1), dim3(1024), 0, st, (const T *)ab, ldab, (int)n,
                           CutSet{(int)kl, (int)(kl + ku + 1), kv, 0}, CutSet{}, 5, 0.0f, flags, host, dinfo);
        BH_LAUNCH_CHECK();
        cut_note(flags, st);
        // (the MFMA kernel's fill of whole columns takes some 30 us to find the
        // gate open, n = 262144; its chains are long enough to wait for the word)
        int r = -1;
        if (tries == 0 && kind != kLuMfma) {
            LuCut<T> seq{};
            seq.flags = flags;
            r = lu_kernel_launch<T>(kind, n, kl, ku, ab, ldab, ipiv, dinfo, st, &seq);
        }
        const int closed = cut_poll(host, st);
        if (r != BH_OK && r != -1) return r;  // -1: not the whole system (its 32-bit offsets), its blocks perhaps
        if (closed < 0) BH_HIP(hipStreamSynchronize(st));
        if (closed != 0) {
            *out = r == BH_OK ? kCutLaunched : kCutNot;
            return BH_OK;
        }
        const unsigned gx = (unsigned)imin(64, cdiv((i64)g.span() * H, 1024));
        hipLaunchKernelGGL(lu_cut_copy<T>, dim3(gx, g.p), dim3(256), 0, st, cut, (const T *)ab, ldab, kv);
        r = lu_kernel_launch<T>(kind, n, kl, ku, cut.ab, H, cut.ipiv, cut.info, st, &cut);
        if (r != BH_OK) return r == -1 ? BH_OK : r;  // -1: the kernel does not take this band
        hipLaunchKernelGGL(lu_cut_check<T>, dim3(g.p), dim3(256), 0, st, cut, kv, (int)up16(kv), flags);
        hipLaunchKernelGGL(lu_cut_commit<T>, dim3(gx, g.p), dim3(256), 0, st, cut, ab, ldab, ipiv, host + 1);
        BH_LAUNCH_CHECK();
        BH_HIP(hipStreamSynchronize(st));
        if (host[1] == 0) {
            *out = kCutDone;
            return BH_OK;
        }
        // long enough that four times the lead-in is still little of the chain: once more
        if (n < 32 * (i64)(g.L + 4 * g.W)) return BH_OK;
    }
    return BH_OK;
}

template <typename T>
static int gbtrf_impl(i64 m, i64 n, i64 kl, i64 ku, T *ab, i64 ldab, i64 *ipiv, i64 *info_host) {
    BH_ARG(m >= 0, 1);
    BH_ARG(n >= 0, 2);
    BH_ARG(kl >= 0, 3);
    BH_ARG(ku >= 0, 4);
    BH_ARG(ldab >= 2 * kl + ku + 1, 6);
    BH_ARG(info_host != nullptr, 8);
    *info_host = 0;
    if (m == 0 || n == 0) return BH_OK;
    i64 *dinfo = nullptr;
    {
        const int cs = ctrl_words(&dinfo);
        if (cs) return cs;
    }
    // register-resident kernel when the window fits one of its shapes,
    // otherwise the barrier-stepped kernel working in global memory
    const int ov = lu_kernel_override();
    int st = -1;
    const bool mfma = ov == 5 || (ov == 0 && ((ku >= 65 && kl >= 32) || (kl >= 8 && ku >= 8 && imin(m, n) >= kLongLu)));
    LuKernel kind = kLuNone;  // the kernel that runs the system, where it has a form for blocks
    const size_t ml = mfma_lds_bytes(kl, sizeof(T));
    if (mfma)
        kind = ml > 0 && ml + 4096 <= 160 * 1024 ? kLuMfma : kLuNone;
    else if (ov == 0 && kl <= 16 && kl + ku <= 63 && !getenv("BANDEDHIP_SMALL_LU"))
        kind = kLuLane;
    else if (ov == 0 && kl >= 16 && blk_shape_for(kl, ku) >= 0)
        kind = kLuBlk;
    CutOutcome cut = kCutNot;
    cut_begin();
    if (m == n && kind != kLuNone) {
        const int cs = gbtrf_cut<T>(kind, n, kl, ku, ab, ldab, ipiv, dinfo, &cut);
        if (cs) return cs;
        if (cut == kCutDone) return BH_OK;
    }
    if (cut == kCutNot) BH_HIP(hipMemsetAsync(dinfo, 0, 2 * sizeof(i64), stream()));
    // The MFMA-blocked factorisation (pivots equal xGBTF2's, factors to
    // rounding): where the reference itself runs blocked xGBTRF (ku >= 65,
    // kl >= 32), and for long systems with kl, ku >= 8, where the one-wave
    // chain of the narrow kernels is the longer path (n = 262144, (16,16):
    // 142 ms against 278 ms).  Shorter narrow systems keep the bit-exact
    // xGBTF2 kernels.
    if (cut == kCutLaunched)
        st = BH_OK;
    else if (mfma)
        st = mfma_gbtrf_launch<T>(m, n, kl, ku, ab, ldab, ipiv, dinfo, stream(), nullptr);
    // The one-wave lane kernel exists for kl <= 16; above 16 the
    // blocked kernel beats the generic one-wave kernel (at n = 65536, (24,24):
    // 113.5 ms against 278.6 ms, identical factors), so it goes first there.
    if (st == -1 && (ov == 4 || (ov == 0 && kl <= 16))) st = small_gbtrf_launch<T>(m, n, kl, ku, ab, ldab, ipiv, dinfo, stream());
    if (st == -1 && (ov == 1 || (ov == 0 && kl >= 16)))
        st = blk_gbtrf_launch<T>(m, n, kl, ku, ab, ldab, ipiv, dinfo, stream(), nullptr);
    if (st == -1 && ov != 3) st = reg_gbtrf_launch<T>(m, n, kl, ku, ab, ldab, ipiv, dinfo, stream());
    if (st == -1) {
        LuSys<T> s{ab, ipiv, m, n, kl, ku, ldab};
        hipLaunchKernelGGL(gbtf2_single<T>, dim3(1), dim3(kLuThreads), 0, stream(), s, dinfo);
        BH_LAUNCH_CHECK();
    } else if (st != BH_OK) {
        return st;
    }
    i64 hinfo[2] = {0, 0};
    BH_HIP(hipMemcpyAsync(hinfo, dinfo, 2 * sizeof(i64), hipMemcpyDeviceToHost, stream()));
    BH_HIP(hipStreamSynchronize(stream()));
    if (hinfo[1] != 0) {
        set_error("gbtrf: an internal wait of the blocked kernel gave up; the factors are not valid");
        return BH_ERR_INTERNAL;
    }
    *info_host = hinfo[0];
    return BH_OK;
}

}  // namespace bh

using namespace bh;

extern "C" {

int bh_dgbtrf(bh_int m, bh_int n, bh_int kl, bh_int ku, double *AB, bh_int ldab, bh_int *ipiv, bh_int *info_host) {
    return gbtrf_impl<double>(m, n, kl, ku, AB, ldab, ipiv, info_host);
}

int bh_sgbtrf(bh_int m, bh_int n, bh_int kl, bh_int ku, float *AB, bh_int ldab, bh_int *ipiv, bh_int *info_host) {
    return gbtrf_impl<float>(m, n, kl, ku, AB, ldab, ipiv, info_host);
}

}  // extern "C"
