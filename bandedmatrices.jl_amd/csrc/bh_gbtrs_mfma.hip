// bh_gbtrs_mfma.hip -- blocked band solve with the factors of bh_?gbtrf,
// panels of PB rows applied on the matrix cores (gfx950 MFMA 16x16x4).
//
// The reference solves with LAPACK.gbtrs! (src/banded/linalg.jl:24-30):
// xGBTRS applies, column by column, the row interchange of step j and the
// rank-1 update of the rows below it (the forward sweep with L), then the
// upper band solve with U (xTBSV).  Both sweeps are a chain of n dependent
// steps.  Here the chain has n/PB links instead:
//
// Forward.  For panel P (rows j0 = P*PB .. j0+PB-1) the window is the RW =
// kl+PB rows its interchanges and multipliers touch.  Applying the PB steps
// of the panel to the window equals (with the panel's row permutation perm,
// its multipliers in final row order L11 (unit lower, PB x PB) and L21
// (kl x PB))
//     Y1 = L11^{-1} (perm W)[0:PB]            the panel's finished rows
//     W' = (perm W)[PB:RW] - L21 Y1           the rows the next panel sees
//        = (perm W)[PB:RW] - M21 (perm W)[0:PB],   M21 = L21 L11^{-1}
// perm, L11^{-1} and M21 depend on the factors only; a parallel pre-pass
// (one workgroup per panel) builds them once per factorisation.  L21 in
// final order is xGBTRF's form of the multipliers before it "partially
// undoes" the interchanges: each stored column c is moved to the positions
// its rows reach after the panel's later interchanges.
// Backward.  Panels from the last: X1 = U11^{-1} Y[j0:j0+PB], and the kv =
// kl+ku rows above the panel lose U[j0-kv:j0, j0:j0+PB] X1 =
// V Y[j0:j0+PB], V = U[j0-kv:j0, j0:j0+PB] U11^{-1}.
//
// Both products of a link read only the window as it stands, so they run
// side by side: one workgroup solves 16 right-hand sides with one MFMA
// product per 16-row tile and one LDS-only barrier per link; the operands
// are loaded two links ahead.  Results equal xGBTRS's to rounding (the
// diagonal blocks through their inverses, a panel's updates in one sum),
// not bit for bit: this solve serves the mixed-precision refinement, whose
// corrections need an accurate solve, not LAPACK's operation order;
// bh_?gbtrs stays the bit-exact path.
//
// Cut systems (bh_cut.hpp).  Where the factors are dominant each sweep runs by
// blocks of panels, one workgroup per block and 16 right-hand sides, B -> Y
// -> Z; the LDS window a block leaves must equal, bit for bit, the one the
// next block has when its own panels begin.
#include <type_traits>

#include "bh_common.hpp"
#include "bh_cut.hpp"
#include "bh_mfma.hpp"

namespace bh {

namespace {

template <typename T>
struct TStride {
    static constexpr int value = sizeof(T) == 4 ? 20 : 18;  // LDS row stride of [rows][16] tiles
};

// Per panel the pre-pass writes one record of A operands, each 16-row tile
// lane-major (lane l's PB/4 K-chunk values contiguous, so a lane loads its
// operands with 16-byte reads): L11^{-1} (PB/16 tiles), M21 (KT tiles),
// U11^{-1} (PB/16 tiles), -V (KTU tiles) -- the update blocks negated, so
// the sweeps accumulate onto the rows' current values; and one record of
// 16-bit window rows, as byte offsets into the forward sweep's LDS window:
// the gather rows of the diagonal-block product (4 x PB/4) and the C-operand
// rows of each M21 tile (KT x 16).
template <typename T, int PB>
struct TrsLayout {
    int n, kl, ku, kv, RW, KT, KTU, np;
    size_t linv_off, l21_off, uinv_off, ublk_off, per_panel;  // elements of T
    size_t cidx_off, idx_u16;                                 // 16-bit entries
    static TrsLayout make(i64 n, i64 kl, i64 ku) {
        TrsLayout L{};
        L.n = (int)n;
        L.kl = (int)kl;
        L.ku = (int)ku;
        L.kv = (int)(kl + ku);
        L.RW = (int)kl + PB;
        L.KT = (int)((kl + 15) / 16);
        L.KTU = (int)((kl + ku + 15) / 16);
        L.np = (int)((n + PB - 1) / PB);
        L.linv_off = 0;
        L.l21_off = (size_t)PB * PB;
        L.uinv_off = L.l21_off + (size_t)L.KT * 16 * PB;
        L.ublk_off = L.uinv_off + (size_t)PB * PB;
        L.per_panel = L.ublk_off + (size_t)L.KTU * 16 * PB;
        L.cidx_off = (size_t)PB;  // 4 x PB/4 gather rows first
        L.idx_u16 = (L.cidx_off + (size_t)L.KT * 16 + 7) & ~(size_t)7;
        return L;
    }
};

constexpr int kTrsTrip = 6;  // panels per trip of the sweeps' loops

// ---------------------------------------------------------------- pre-pass
// One workgroup per panel: perm, L11^{-1} and L21 in final row order, U11^{-1},
// the matrices stored in MFMA A-operand order (16x4 blocks, lane i+16k holding
// element (i, k)), so the solve kernels load them with one coalesced read each.
template <typename T, int PB>
__global__ __launch_bounds__(256) void trs_prep(const T *__restrict__ ab, i64 ldab, const i64 *__restrict__ ipiv,
                                                TrsLayout<T, PB> L, unsigned short *__restrict__ idxA,
                                                T *__restrict__ rec) {
    extern __shared__ __align__(16) unsigned char tp_raw[];
    constexpr int LS = PB + 1;
    const int RW = L.RW, n = L.n, kl = L.kl, kv = L.kv;
    const int top = 16 * L.KTU;
    T *Lf = reinterpret_cast<T *>(tp_raw);  // RW x LS
    T *Ut = Lf + (size_t)RW * LS;           // PB x LS
    T *Xi = Ut + PB * LS;                   // PB x LS
    T *Xu = Xi + PB * LS;                   // PB x LS
    T *Ub = Xu + PB * LS;                   // top x LS: U block above the panel
    int *perm = reinterpret_cast<int *>(Ub + (size_t)top * LS);
    __shared__ int q[PB];
    const int p = blockIdx.x, tid = threadIdx.x;
    const int j0 = p * PB, nb = min(PB, n - j0);
    for (int e = tid; e < RW * LS; e += 256) Lf[e] = T(0);
    for (int r = tid; r < RW; r += 256) perm[r] = r;
    if (tid < PB) {
        int qq = tid;
        if (tid < nb) {
            const i64 piv = ipiv[j0 + tid] - 1 - j0;  // 0 <= piv - tid <= kl for valid factors
            qq = (piv >= tid && piv < RW) ? (int)piv : tid;
        }
        q[tid] = qq;
    }
    __syncthreads();
    if (tid == 0) {
        for (int c = 0; c < nb; ++c) {
            const int a = perm[c];
            perm[c] = perm[q[c]];
            perm[q[c]] = a;
        }
    }
    // multipliers of column c sit at positions c+1..c+kl after step c; the
    // later interchanges of the panel carry position r on.  Every thread
    // follows its own entries through them (with a barrier per column, each
    // waited for its column's load).  2048 panels, (128,128), FP32: 455 -> 420 us
    // with that, 257 with the inverses in registers and the products below
    // eight chunks to a thread.  (U's block read along its columns instead
    // cost 25 us: its LDS writes then conflict.)
    const bool moved = __syncthreads_or(tid < PB && q[tid < PB ? tid : 0] != tid);
    for (int e = tid; e < nb * kl; e += 256) {
        const int c = e / kl, r = c + 1 + e - c * kl;
        if (r < RW && j0 + r < n) {
            const T v = ab[(i64)(j0 + c) * ldab + (kv + r - c)];
            int f = r;
            if (moved)
                for (int s = c + 1; s < nb; ++s) f = f == s ? q[s] : f == q[s] ? s : f;
            Lf[f * LS + c] = v;
        }
    }
    __syncthreads();
    if (tid < PB) Lf[tid * LS + tid] = T(1);
    // U11 (upper, identity past the last column)
    for (int e = tid; e < PB * PB; e += 256) {
        const int i = e / PB, j = e - i * PB;
        T v = T(0);
        if (j >= nb)
            v = (i == j) ? T(1) : T(0);
        else if (i <= j && j - i <= kv)
            v = ab[(i64)(j0 + j) * ldab + (kv + i - j)];
        Ut[i * LS + j] = v;
    }
    __syncthreads();
    // U(i, j) above the panel: i = j0 - top + r, j = j0 + c
    for (int e = tid; e < top * PB; e += 256) {
        const int r = e / PB, c = e - r * PB;
        const int i = j0 - top + r, j = j0 + c, d = kv + i - j;
        Ub[r * LS + c] = (i >= 0 && j < n && d >= 0) ? ab[(i64)j * ldab + d] : T(0);
    }
    // The inverses, one column to a thread, in registers and fully unrolled:
    // L11^{-1} by forward substitution on the first wave, U11^{-1} by back
    // substitution on the second.
    if (tid < PB) {
        const int j = tid;
        T X[PB];
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            T s = T(0);
#pragma unroll
            for (int k = 0; k < i; ++k) {
                const T f = dfma(Lf[i * LS + k], X[k], s);
                s = k >= j ? f : s;
            }
            X[i] = i > j ? -s : (i == j ? T(1) : T(0));
            Xi[i * LS + j] = X[i];
        }
    } else if (tid >= 64 && tid < 64 + PB) {
        const int j = tid - 64;
        T X[PB];
#pragma unroll
        for (int i = PB - 1; i >= 0; --i) {
            T s = (i == j) ? T(1) : T(0);
#pragma unroll
            for (int k = i + 1; k < PB; ++k) {
                const T f = dfma(-Ut[i * LS + k], X[k], s);
                s = k <= j ? f : s;
            }
            X[i] = i <= j ? s / Ut[i * LS + i] : T(0);
            Xu[i * LS + j] = X[i];
        }
    }
    __syncthreads();
    constexpr int NS = PB / 4;
    T *out = rec + (size_t)p * L.per_panel;
    // element e of a tile block: tile e / (64 NS), lane (e / NS) % 64, chunk e % NS
    for (int e = tid; e < PB * PB; e += 256) {
        const int s = e % NS, lane = (e / NS) & 63, ti = e / (64 * NS);
        const int at = (16 * ti + (lane & 15)) * LS + 4 * s + (lane >> 4);
        out[L.linv_off + e] = Xi[at];
        out[L.uinv_off + e] = Xu[at];
    }
    // -M21 = -L21 L11^{-1} and -V = -U_block U11^{-1}, stored negated (the sweeps
    // accumulate onto the C operand): a thread forms the NS chunks of one
    // lane's row together, the inverse's triangle kept by selects
    auto product = [&](const T *A, int rows, const T *X, bool low, int tiles, size_t off) {
        for (int e = tid; e < tiles * 64; e += 256) {
            const int lane = e & 63, r = 16 * (e >> 6) + (lane & 15), kq = lane >> 4;
            const T *row = A + min(r, rows - 1) * LS;
            T acc[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) acc[s] = T(0);
#pragma unroll 8
            for (int k = 0; k < PB; ++k) {
                const T a = row[k];
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int c = 4 * s + kq;
                    const T f = dfma(a, X[k * LS + c], acc[s]);
                    acc[s] = (low ? k >= c : k <= c) ? f : acc[s];
                }
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) out[off + (size_t)e * NS + s] = r < rows ? -acc[s] : -T(0);
        }
    };
    product(Lf + PB * LS, RW - PB, Xi, true, L.KT, L.l21_off);
    product(Ub, top, Xu, false, L.KTU, L.ublk_off);
    unsigned short *ix = idxA + (size_t)p * L.idx_u16;
    // window rows as LDS byte offsets of the sweep's [rows][SW] buffer (< 2^16)
    constexpr int RB_ = TStride<T>::value * (int)sizeof(T);
    for (int e = tid; e < PB; e += 256) ix[e] = (unsigned short)(perm[4 * (e % NS) + e / NS] * RB_);  // [kq][s]
    for (int e = tid; e < L.KT * 16; e += 256) {
        const int v = e & 3, kq = (e >> 2) & 3, t = e >> 4;
        ix[L.cidx_off + e] = (unsigned short)(perm[min(PB + 16 * t + drow<T>(kq, v), RW - 1)] * RB_);
    }
}

// Operands of one panel, loaded two panels ahead of their use (three sets
// rotate), so the load latency is hidden behind two panels of work.  Every
// wave issues the same buffer loads and stores in every panel (clamped
// indices; out-of-range offsets read 0 and drop stores), so the compiler's
// wait counts stay exact: a panel waits only for loads two panels old.
template <typename T, int NS, int MT>
struct PanelOps {
    T a[NS];       // A operands of the diagonal-block product
    T b[MT][NS];   // A operands of this wave's update tiles
    int g[NS];     // forward: window rows gathered as B operands (rows 4s+kq)
    int c[MT][4];  // forward: window rows of the update tiles' C operands
    T fresh;       // one element of the rows entering the window
};

typedef unsigned trs_v4u __attribute__((ext_vector_type(4)));
typedef unsigned trs_v2u __attribute__((ext_vector_type(2)));

// N consecutive elements at byte offset off (16-byte aligned) with 16-byte loads
template <typename T, int N>
__device__ __forceinline__ void bload_vec(__amdgpu_buffer_rsrc_t r, int off, T (&dst)[N]) {
    static_assert((N * sizeof(T)) % 16 == 0, "whole 16-byte loads");
#pragma unroll
    for (int q = 0; q < (int)(N * sizeof(T) / 16); ++q) {
        const trs_v4u x = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16 * q, 0, 0);
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // through a scalar: __builtin_bit_cast of a vector element
                // (x[i] directly) is lowered wrongly by this compiler
                const unsigned e = x[i];
                dst[4 * q + i] = __builtin_bit_cast(float, e);
            }
        } else {
            dst[2 * q] = __builtin_bit_cast(double, (trs_v2u){x[0], x[1]});
            dst[2 * q + 1] = __builtin_bit_cast(double, (trs_v2u){x[2], x[3]});
        }
    }
}

// ---------------------------------------------------------------- forward sweep
// B (n x nrhs, ldb) <- L^{-1} P B for the 16 columns starting at 16*blockIdx.x.
// LDS addresses are precomputed per lane; the window buffer a panel reads
// (cur) is a compile-time constant of each of the six unrolled panels.
// By blocks (cut.g.p > 0) it reads B and writes Y (the same array otherwise).
template <typename T, int PB, int NW, int MT>
__global__ __launch_bounds__(64 * NW) void trs_fwd(const T *B, i64 ldb, T *Y, i64 ldy, int nrhs, TrsLayout<T, PB> L,
                                                   const unsigned short *idxA, const T *rec, SweepCut<T> cut) {
    const int blk = blockIdx.y;
    if (cut.g.p > 0 ? cut_closed(cut.flags) : (cut.flags && !cut_failed(cut.flags))) return;
    // panels p0 .. p1-1, its own from pown: multiples of the trip of six
    const int p0 = cut.g.p > 0 ? kTrsTrip * cut.g.start(blk) : 0, pown = cut.g.p > 0 ? kTrsTrip * cut.g.own(blk) : 0;
    const int p1 = cut.g.p > 0 ? min(kTrsTrip * cut.g.end(blk), L.np) : L.np;
    using v4 = typename Mf<T>::v4;
    constexpr int SW = TStride<T>::value;
    constexpr int NS = PB / 4;   // K chunks of a panel product
    constexpr int NP = PB / 16;  // 16-row tiles of a panel (MT: M21 tiles per wave)
    constexpr int ES = (int)sizeof(T);
    constexpr int RS = SW * ES;  // LDS bytes per window row
    static_assert(NS == 8, "the gather rows of a lane are one 16-byte load");
    using Ops = PanelOps<T, NS, MT>;
    extern __shared__ __align__(16) unsigned char tf_raw[];
    const int RW = L.RW, KT = L.KT, n = L.n, np = L.np;
    const int RWP = 16 * ((RW + 15) / 16) + 1;  // + one dump row for results past RW
    const int WB = RWP * RS;                    // bytes of one window buffer
    // w is wave-uniform (branches on it stay scalar)
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int jc = lane & 15, kq = lane >> 4;
    const int fr = tid >> 4, fj = tid & 15;  // PB*16 <= 64*NW threads carry one fresh element
    const int c0 = 16 * blockIdx.x;
    const bool colok = c0 + jc < nrhs;
    const __amdgpu_buffer_rsrc_t rB = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(B) + (i64)c0 * ldb, 0,
                                                                        (int)(16 * ldb * ES), kQRsrcWord3);
    const __amdgpu_buffer_rsrc_t rY = __builtin_amdgcn_make_buffer_rsrc(Y + (i64)c0 * ldy, 0, (int)(16 * ldy * ES),
                                                                        kQRsrcWord3);
    // per-lane byte offsets inside a panel's records
    const int offA = (int)((L.linv_off + ((size_t)min(w, NP - 1) * 64 + lane) * NS) * ES);
    int offB[MT], offC[MT], wdst[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int t = min(w + m * NW, KT - 1);
        offB[m] = (int)((L.l21_off + ((size_t)t * 64 + lane) * NS) * ES);
        offC[m] = (int)((L.cidx_off + (size_t)(t * 4 + kq) * 4) * 2);
#pragma unroll
        for (int v = 0; v < 4; ++v) {  // where row r = PB + 16t + drow lands in the next window
            const int r = PB + 16 * (w + m * NW) + drow<T>(kq, v);
            wdst[m][v] = (r < RW ? r - PB : RWP - 1) * RS + jc * ES;
        }
    }
    const int fdst = fr < PB ? (RW - PB + fr) * RS + fj * ES : (RWP - 1) * RS + fj * ES;
    // Y1 rows of this lane relative to the panel (stores of waves past NP
    // and of columns past nrhs go out of range)
    int ysto[4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
        ysto[v] = (w < NP && colok) ? (jc * (int)ldy + 16 * w + drow<T>(kq, v)) * ES : kQOob;

    auto issue = [&](int p, Ops &o) {
        const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T *>(rec) + (size_t)p * L.per_panel, 0, (int)(L.per_panel * ES), kQRsrcWord3);
        const __amdgpu_buffer_rsrc_t ri = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<unsigned short *>(idxA) + (size_t)p * L.idx_u16, 0, (int)(L.idx_u16 * 2), kQRsrcWord3);
        bload_vec<T, NS>(rr, offA, o.a);
#pragma unroll
        for (int m = 0; m < MT; ++m) bload_vec<T, NS>(rr, offB[m], o.b[m]);
        const trs_v4u gi = __builtin_amdgcn_raw_buffer_load_b128(ri, kq * NS * 2, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o.g[2 * q] = (int)(gi[q] & 0xffffu);
            o.g[2 * q + 1] = (int)(gi[q] >> 16);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const trs_v2u ci = __builtin_amdgcn_raw_buffer_load_b64(ri, offC[m], 0, 0);
            o.c[m][0] = (int)(ci[0] & 0xffffu);
            o.c[m][1] = (int)(ci[0] >> 16);
            o.c[m][2] = (int)(ci[1] & 0xffffu);
            o.c[m][3] = (int)(ci[1] >> 16);
        }
        const int row = p * PB + RW + fr;
        o.fresh = qbload<T>(rB, (fr < PB && row < n && c0 + fj < nrhs) ? (fj * (int)ldb + row) * ES : kQOob);
    };

    unsigned char *lds = tf_raw;
    // one panel: uses `u`, starts the loads of panel p+2 into `ld`
    auto panel = [&](int p, auto curc, const Ops &u, Ops &ld) {
        constexpr int cur = decltype(curc)::value;
        const int j0 = p * PB;
        const unsigned char *Wc = lds + cur * WB + jc * ES;
        unsigned char *Wn = lds + (cur ^ 1) * WB;
        issue(min(p + 2, np - 1), ld);
        // the gathered rows (perm W)[0:PB] as B operands
        T g0[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) g0[s] = *reinterpret_cast<const T *>(Wc + u.g[s]);
        // W' = (perm W)[PB:RW] + (-M21) (perm W)[0:PB]
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int t = w + m * NW;
            if (t < KT) {
                v4 z;
#pragma unroll
                for (int v = 0; v < 4; ++v) z[v] = *reinterpret_cast<const T *>(Wc + u.c[m][v]);
#pragma unroll
                for (int s = 0; s < NS; ++s) z = Mf<T>::mma(u.b[m][s], g0[s], z);
#pragma unroll
                for (int v = 0; v < 4; ++v) *reinterpret_cast<T *>(Wn + wdst[m][v]) = z[v];
            }
        }
        *reinterpret_cast<T *>(Wn + fdst) = u.fresh;
        // Y1 = L11^{-1} (perm W)[0:PB], to B (rows past n, columns past
        // nrhs and waves past NP: dropped)
        v4 y = {T(0), T(0), T(0), T(0)};
        if (w < NP) {
#pragma unroll
            for (int s = 0; s < NS; ++s) y = Mf<T>::mma(u.a[s], g0[s], y);
        }
        const bool full = j0 + PB <= n;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * w + drow<T>(kq, v);
            const int off = (full || j0 + r < n) && p >= pown && ysto[v] != kQOob ? ysto[v] + j0 * ES : kQOob;
            qbstore<T>(rY, off, y[v]);
        }
        lds_barrier();
    };

    Ops S0, S1, S2;
    issue(p0, S0);
    issue(min(p0 + 1, np - 1), S1);
    // window of the first panel (buffer 0)
    for (int e = tid; e < (RWP - 1) * 16; e += 64 * NW) {
        const int r = e >> 4, j = e & 15, row = p0 * PB + r;
        *reinterpret_cast<T *>(lds + r * RS + j * ES) =
            qbload<T>(rB, (r < RW && row < n && c0 + j < nrhs) ? (j * (int)ldb + row) * ES : kQOob);
    }
    lds_barrier();
    // the window (buffer 0 between trips) for the seam check; rows past RW hold nothing
    auto keep = [&](int which) {
        T *d = cut.at(blk, which, RW * 16);
        for (int e = tid; e < RW * 16; e += 64 * NW)
            d[e] = *reinterpret_cast<const T *>(lds + (e >> 4) * RS + (e & 15) * ES);
    };
    // six panels per trip (three operand sets x two window buffers); panels
    // past the last store nothing: their rows are past n
    const std::integral_constant<int, 0> b0;
    const std::integral_constant<int, 1> b1;
    for (int p = p0; p < p1; p += kTrsTrip) {
        if (blk > 0 && p == pown) {
            keep(0);
            lds_barrier();
        }
        panel(p, b0, S0, S2);
        panel(p + 1, b1, S1, S0);
        panel(p + 2, b0, S2, S1);
        panel(p + 3, b1, S0, S2);
        panel(p + 4, b0, S1, S0);
        panel(p + 5, b1, S2, S1);
    }
    if (blk + 1 < cut.g.p) keep(1);
}

// ---------------------------------------------------------------- backward sweep
// B <- U^{-1} B (U: upper band of width kv = kl+ku) for 16 columns; the U
// operands come from the pre-pass records.
// By blocks it reads B and writes X (the same array otherwise).
template <typename T, int PB, int NW, int MT>
__global__ __launch_bounds__(64 * NW) void trs_bwd(const T *B, i64 ldb, T *X, i64 ldx, int nrhs, TrsLayout<T, PB> L,
                                                   const T *rec, int RB, SweepCut<T> cut) {
    const int blk = blockIdx.y;
    if (cut.g.p > 0 ? cut_closed(cut.flags) : (cut.flags && !cut_failed(cut.flags))) return;
    // panels by their index from the last one: q0 .. q1-1, its own from qown
    const int q0 = cut.g.p > 0 ? kTrsTrip * cut.g.start(blk) : 0, qown = cut.g.p > 0 ? kTrsTrip * cut.g.own(blk) : 0;
    const int q1 = cut.g.p > 0 ? min(kTrsTrip * cut.g.end(blk), L.np) : L.np;
    using v4 = typename Mf<T>::v4;
    constexpr int SW = TStride<T>::value;
    constexpr int NS = PB / 4;
    constexpr int NP = PB / 16;  // (MT: V tiles per wave)
    constexpr int ES = (int)sizeof(T);
    constexpr int RS = SW * ES;
    using Ops = PanelOps<T, NS, MT>;
    extern __shared__ __align__(16) unsigned char tb_raw[];
    const int n = L.n, KTU = L.KTU, np = L.np;
    const int top = 16 * KTU;  // rows above a panel that it updates (>= kv)
    unsigned char *Yr = tb_raw;  // ring [RB][SW], row i in slot i & (RB-1)
    const int msk = RB - 1;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int jc = lane & 15, kq = lane >> 4;
    const int fr = tid >> 4, fj = tid & 15;
    const int c0 = 16 * blockIdx.x;
    const bool colok = c0 + jc < nrhs;
    const __amdgpu_buffer_rsrc_t rB = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(B) + (i64)c0 * ldb, 0,
                                                                        (int)(16 * ldb * ES), kQRsrcWord3);
    const __amdgpu_buffer_rsrc_t rX = __builtin_amdgcn_make_buffer_rsrc(X + (i64)c0 * ldx, 0, (int)(16 * ldx * ES),
                                                                        kQRsrcWord3);
    const int offA = (int)((L.uinv_off + ((size_t)min(w, NP - 1) * 64 + lane) * NS) * ES);
    int offB[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
        offB[m] = (int)((L.ublk_off + ((size_t)min(w + m * NW, KTU - 1) * 64 + lane) * NS) * ES);
    // lane parts of the ring addresses: B operand rows 4s+kq, result rows drow(kq, v)
    const int yb = kq * RS + jc * ES;
    int zb[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) zb[v] = drow<T>(kq, v) * RS + jc * ES;
    int xsto[4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
        xsto[v] = (w < NP && colok) ? (jc * (int)ldx + 16 * w + drow<T>(kq, v)) * ES : kQOob;

    auto issue = [&](int p, Ops &o) {
        const int j0 = p * PB;
        const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T *>(rec) + (size_t)p * L.per_panel, 0, (int)(L.per_panel * ES), kQRsrcWord3);
        bload_vec<T, NS>(rr, offA, o.a);
#pragma unroll
        for (int m = 0; m < MT; ++m) bload_vec<T, NS>(rr, offB[m], o.b[m]);
        const int frow = j0 - top - PB + fr;
        o.fresh = qbload<T>(rB, (fr < PB && frow >= 0 && c0 + fj < nrhs) ? (fj * (int)ldb + frow) * ES : kQOob);
    };

    // panel index q counts from the last panel (q = 0 is panel np-1).  Ring
    // slots of negative rows (first panels) take throwaway updates: they are
    // never read, as RB >= top + 2 PB keeps them clear of live rows.
    auto panel = [&](int q, const Ops &u, Ops &ld) {
        const int p = np - 1 - q;
        const int j0 = p * PB;
        issue(max(p - 2, 0), ld);
        // Y[j0:j0+PB] as B operands (j0 & msk is a multiple of PB: no wrap inside)
        const unsigned char *yrow = Yr + (j0 & msk) * RS + yb;
        T y0[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) y0[s] = *reinterpret_cast<const T *>(yrow + 4 * s * RS);
        // Y[j0-top : j0] += (-V) Y[j0:j0+PB]
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int t = w + m * NW;
            if (t < KTU) {
                unsigned char *zrow = Yr + ((j0 - top + 16 * t) & msk) * RS;
                v4 z;
#pragma unroll
                for (int v = 0; v < 4; ++v) z[v] = *reinterpret_cast<const T *>(zrow + zb[v]);
#pragma unroll
                for (int s = 0; s < NS; ++s) z = Mf<T>::mma(u.b[m][s], y0[s], z);
#pragma unroll
                for (int v = 0; v < 4; ++v) *reinterpret_cast<T *>(zrow + zb[v]) = z[v];
            }
        }
        const int frow = j0 - top - PB + fr;
        if (fr < PB && frow >= 0) *reinterpret_cast<T *>(Yr + (frow & msk) * RS + fj * ES) = u.fresh;
        // X1 = U11^{-1} Y[j0:j0+PB], to B
        v4 x = {T(0), T(0), T(0), T(0)};
        if (w < NP) {
#pragma unroll
            for (int s = 0; s < NS; ++s) x = Mf<T>::mma(u.a[s], y0[s], x);
        }
        const bool full = j0 >= 0 && j0 + PB <= n;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * w + drow<T>(kq, v);
            const int off =
                (full || (j0 + r >= 0 && j0 + r < n)) && q >= qown && xsto[v] != kQOob ? xsto[v] + j0 * ES : kQOob;
            qbstore<T>(rX, off, x[v]);
        }
        lds_barrier();
    };

    Ops S0, S1, S2;
    issue(np - 1 - q0, S0);
    issue(max(np - 2 - q0, 0), S1);
    // ring: rows [jl - top, jl + PB) of the first panel taken (zero past n)
    const int jl = (np - 1 - q0) * PB;
    for (int e = tid; e < (top + PB) * 16; e += 64 * NW) {
        const int rr = e >> 4, j = e & 15;
        const int row = jl - top + rr;
        *reinterpret_cast<T *>(Yr + (row & msk) * RS + j * ES) =
            qbload<T>(rB, (row >= 0 && row < n && c0 + j < nrhs) ? (j * (int)ldb + row) * ES : kQOob);
    }
    lds_barrier();
    // panels before the first (at most two) touch only negative rows: their
    // stores are dropped and their ring updates land in throwaway slots
    // rows [j0 - top, j0 + PB) of panel q for the seam check
    auto keep = [&](int which, int q) {
        const int base = (np - 1 - q) * PB - top;
        T *d = cut.at(blk, which, (top + PB) * 16);
        for (int e = tid; e < (top + PB) * 16; e += 64 * NW) {
            const int row = base + (e >> 4);
            d[e] = row >= 0 ? *reinterpret_cast<const T *>(Yr + (row & msk) * RS + (e & 15) * ES) : T(0);
        }
    };
    for (int q = q0; q < q1; q += 3) {
        if (blk > 0 && q == qown) {
            keep(0, q);
            lds_barrier();
        }
        panel(q, S0, S2);
        panel(q + 1, S1, S0);
        panel(q + 2, S2, S1);
    }
    if (blk + 1 < cut.g.p) keep(1, q1);
}

constexpr int kTrsPB = 32;
constexpr int kTrsNW = 8;

// Blocks of a sweep with bandwidth k, in trips of six panels: the lead-in of
// sweep_geom (20 k rows in FP64, 10 k in FP32, and the window itself); at most
// 512 workgroups over all groups of 16 right-hand sides, and own trips of at
// least a quarter of the lead-in (every block reads its lead-in's records again).
template <typename T>
CutGeom trs_geom(int np, i64 k, i64 groups) {
    const int rows = kTrsTrip * kTrsPB;
    const i64 G = cdiv(np, kTrsTrip), W = cdiv((sizeof(T) == 8 ? 20 : 10) * k, rows) + cdiv(k + kTrsPB, rows);
    const i64 L = imax(cdiv(G, imax(1, 512 / groups)), (W + 3) / 4);
    CutGeom g{(int)G, (int)L, (int)W, (int)cdiv(G, L)};
    if (2 * (L + W) > G || groups > 65535 || g.p < 2 || g.p > 65535) g.p = 0;
    return g;
}

}  // namespace

// Bytes of the pre-pass output for (n, kl, ku): 0 when the blocked solve does
// not apply (then the caller uses bh_?gbtrs).
template <typename T>
size_t trs_blocked_bytes(i64 n, i64 kl, i64 ku) {
    using Lt = TrsLayout<T, kTrsPB>;
    constexpr int SW = TStride<T>::value;
    // 16 columns of B (leading dimension >= n) must fit one 31-bit buffer offset range
    if (n <= 0 || kl < 1 || 16 * n * (i64)sizeof(T) >= kQOob) return 0;
    // update tiles per wave that the registers hold without spilling:
    // FP32 3 forward, 4 backward; FP64 1 forward, 2 backward
    const i64 mtf = sizeof(T) == 4 ? 3 : 1, mtb = sizeof(T) == 4 ? 4 : 2;
    if (kl > 16 * mtf * kTrsNW || kl + ku > 16 * mtb * kTrsNW) return 0;
    const Lt L = Lt::make(n, kl, ku);
    const int RWP = 16 * ((L.RW + 15) / 16) + 1;
    const size_t fwd_lds = (size_t)(2 * RWP) * SW * sizeof(T);
    int RB = 1;
    while (RB < 16 * L.KTU + 2 * kTrsPB) RB <<= 1;
    const size_t bwd_lds = (size_t)RB * SW * sizeof(T);
    const size_t prep_lds = ((size_t)(L.RW + 3 * kTrsPB + 16 * L.KTU) * (kTrsPB + 1)) * sizeof(T) + L.RW * sizeof(int);
    if (fwd_lds > 160 * 1024 || bwd_lds > 160 * 1024 || prep_lds > 160 * 1024) return 0;
    const size_t recs = (size_t)L.np * L.per_panel * sizeof(T);
    const size_t idxs = (size_t)L.np * L.idx_u16 * 2;
    if (L.per_panel * sizeof(T) >= (size_t)kQOob) return 0;
    return ((recs + 255) & ~(size_t)255) + ((idxs + 255) & ~(size_t)255);
}

template <typename T>
int trs_blocked_prepare(i64 n, i64 kl, i64 ku, const T *ab, i64 ldab, const i64 *ipiv, void *work, hipStream_t st) {
    using Lt = TrsLayout<T, kTrsPB>;
    const Lt L = Lt::make(n, kl, ku);
    const size_t recs = (size_t)L.np * L.per_panel * sizeof(T);
    T *rec = (T *)work;
    unsigned short *idx = (unsigned short *)((char *)work + ((recs + 255) & ~(size_t)255));
    const size_t lds = ((size_t)(L.RW + 3 * kTrsPB + 16 * L.KTU) * (kTrsPB + 1)) * sizeof(T) + L.RW * sizeof(int);
    auto kern = trs_prep<T, kTrsPB>;
    if (lds > 64 * 1024)
        BH_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)L.np), dim3(256), lds, st, ab, ldab, ipiv, L, idx, rec);
    BH_LAUNCH_CHECK();
    return BH_OK;
}

template <typename T>
int trs_blocked_solve(i64 n, i64 kl, i64 ku, i64 nrhs, const T *ab, i64 ldab, const void *work, T *B, i64 ldb,
                      hipStream_t st) {
    using Lt = TrsLayout<T, kTrsPB>;
    constexpr int SW = TStride<T>::value;
    if (nrhs <= 0 || n <= 0) return BH_OK;
    if (16 * ldb * (i64)sizeof(T) >= kQOob) {
        set_error("gbtrs_blocked: ldb = %lld is too large for 16 columns in one buffer range", (long long)ldb);
        return BH_ERR_WORKSPACE;
    }
    const Lt L = Lt::make(n, kl, ku);
    const size_t recs = (size_t)L.np * L.per_panel * sizeof(T);
    const T *rec = (const T *)work;
    const unsigned short *idx = (const unsigned short *)((const char *)work + ((recs + 255) & ~(size_t)255));
    const dim3 grid((unsigned)((nrhs + 15) / 16));
    const int RWP = 16 * ((L.RW + 15) / 16) + 1;
    const size_t fl = (size_t)(2 * RWP) * SW * sizeof(T);
    const int mtf = (L.KT + kTrsNW - 1) / kTrsNW;
    void (*kf)(const T *, i64, T *, i64, int, Lt, const unsigned short *, const T *, SweepCut<T>) = nullptr;
    if constexpr (sizeof(T) == 4) {
        if (mtf > 3) return BH_ERR_WORKSPACE;
        kf = mtf <= 1 ? trs_fwd<T, kTrsPB, kTrsNW, 1>
           : mtf == 2 ? trs_fwd<T, kTrsPB, kTrsNW, 2>
                      : trs_fwd<T, kTrsPB, kTrsNW, 3>;
    } else {
        if (mtf > 1) return BH_ERR_WORKSPACE;
        kf = trs_fwd<T, kTrsPB, kTrsNW, 1>;
    }
    if (fl > 64 * 1024) BH_HIP(hipFuncSetAttribute((const void *)kf, hipFuncAttributeMaxDynamicSharedMemorySize, (int)fl));
    int RB = 1;
    while (RB < 16 * L.KTU + 2 * kTrsPB) RB <<= 1;
    const size_t bl = (size_t)RB * SW * sizeof(T);
    const int mtb = (L.KTU + kTrsNW - 1) / kTrsNW;
    void (*kb)(const T *, i64, T *, i64, int, Lt, const T *, int, SweepCut<T>) = nullptr;
    if constexpr (sizeof(T) == 4) {
        kb = mtb <= 1 ? trs_bwd<T, kTrsPB, kTrsNW, 1>
           : mtb == 2 ? trs_bwd<T, kTrsPB, kTrsNW, 2>
           : mtb == 3 ? trs_bwd<T, kTrsPB, kTrsNW, 3>
                      : trs_bwd<T, kTrsPB, kTrsNW, 4>;
    } else {
        if (mtb > 2) return BH_ERR_WORKSPACE;
        kb = mtb <= 1 ? trs_bwd<T, kTrsPB, kTrsNW, 1> : trs_bwd<T, kTrsPB, kTrsNW, 2>;
    }
    if (bl > 64 * 1024) BH_HIP(hipFuncSetAttribute((const void *)kb, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bl));
    // By blocks (gate as in bh_gbtrs_ring.hpp), and behind them the whole
    // sweeps, which do nothing where the blocks agreed.  16 right-hand sides,
    // n = 65536, (128,128), FP32: 4.2 -> 0.3 ms, bounded by the W + L links of one block.
    const dim3 block(64 * kTrsNW);
    const CutGeom gl = trs_geom<T>(L.np, kl, grid.x), gu = trs_geom<T>(L.np, kl + ku, grid.x);
    SweepCut<T> cut{};
    char *ws = nullptr;
    cut_begin();
    if (gl.p > 0 && gu.p > 0 && 16 * n * (i64)sizeof(T) < kQOob && cut_enabled()) {
        auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
        const i64 cols = 16 * (i64)grid.x;  // whole groups of 16 columns
        const int cl = L.RW * 16, cu = (16 * L.KTU + kTrsPB) * 16;
        const size_t by = al((size_t)n * cols * sizeof(T)), sl = al((size_t)gl.p * grid.x * 2 * cl * sizeof(T));
        const size_t su = al((size_t)gu.p * grid.x * 2 * cu * sizeof(T));
        ws = (char *)cut_alloc(2 * by + sl + su + 256, st);
        if (ws) {
            T *Y = (T *)ws, *Z = (T *)(ws + by), *snl = (T *)(ws + 2 * by), *snu = (T *)(ws + 2 * by + sl);
            int *flags = (int *)(ws + 2 * by + sl + su);
            const int kd = (int)(kl + ku);
            hipLaunchKernelGGL(cut_gate<T>, dim3(1), dim3(1024), 0, st, ab, ldab, (int)n, CutSet{0, kd + 1, kd, 0},
                               CutSet{kd, (int)kl + 1, kd, 1}, 5, 0.0f, flags, (int *)nullptr, (i64 *)nullptr);
            hipLaunchKernelGGL(kf, dim3(grid.x, gl.p), block, fl, st, (const T *)B, ldb, Y, n, (int)nrhs, L, idx, rec,
                               SweepCut<T>{gl, flags, snl});
            hipLaunchKernelGGL(sweep_check<T>, dim3(gl.p - 1, grid.x), dim3(256), 0, st, (const T *)snl, cl, flags);
            hipLaunchKernelGGL(kb, dim3(grid.x, gu.p), block, bl, st, (const T *)Y, n, Z, n, (int)nrhs, L, rec, RB,
                               SweepCut<T>{gu, flags, snu});
            hipLaunchKernelGGL(sweep_check<T>, dim3(gu.p - 1, grid.x), dim3(256), 0, st, (const T *)snu, cu, flags);
            hipLaunchKernelGGL(sweep_commit<T>, dim3((unsigned)cdiv(n, 256), (unsigned)nrhs), dim3(256), 0, st, (int)n,
                               (const T *)Z, B, 1, ldb, (const int *)flags, (int *)nullptr);
            cut_note(flags, st);
            cut.flags = flags;
        }
    }
    hipLaunchKernelGGL(kf, grid, block, fl, st, (const T *)B, ldb, B, ldb, (int)nrhs, L, idx, rec, cut);
    hipLaunchKernelGGL(kb, grid, block, bl, st, (const T *)B, ldb, B, ldb, (int)nrhs, L, rec, RB, cut);
    const hipError_t e = hipGetLastError();
    cut_free(ws, st);
    return e == hipSuccess ? BH_OK : hip_fail(e, "gbtrs_blocked", __FILE__, __LINE__);
}

template size_t trs_blocked_bytes<float>(i64, i64, i64);
template size_t trs_blocked_bytes<double>(i64, i64, i64);
template int trs_blocked_prepare<float>(i64, i64, i64, const float *, i64, const i64 *, void *, hipStream_t);
template int trs_blocked_prepare<double>(i64, i64, i64, const double *, i64, const i64 *, void *, hipStream_t);
template int trs_blocked_solve<float>(i64, i64, i64, i64, const float *, i64, const void *, float *, i64, hipStream_t);
template int trs_blocked_solve<double>(i64, i64, i64, i64, const double *, i64, const void *, double *, i64,
                                       hipStream_t);

}  // namespace bh

using namespace bh;

template <typename T>
static int gbtrs_blocked_impl(i64 n, i64 kl, i64 ku, i64 nrhs, const T *ab, i64 ldab, const i64 *ipiv, T *B, i64 ldb,
                              void *work, size_t lwork) {
    BH_ARG(n >= 0, 1);
    BH_ARG(kl >= 0, 2);
    BH_ARG(ku >= 0, 3);
    BH_ARG(nrhs >= 0, 4);
    BH_ARG(ldab >= 2 * kl + ku + 1, 6);
    BH_ARG(ldb >= imax(1, n), 9);
    if (n == 0 || nrhs == 0) return BH_OK;
    const size_t need = trs_blocked_bytes<T>(n, kl, ku);
    if (need == 0) {
        set_error("gbtrs_blocked: bands (%lld,%lld) are outside the blocked solve's range (FP32: 1 <= kl <= 384, "
                  "kl+ku <= 512; FP64: 1 <= kl <= 128, kl+ku <= 256); use bh_?gbtrs", (long long)kl, (long long)ku);
        return BH_ERR_WORKSPACE;
    }
    if (work == nullptr || lwork < need) {
        set_error("gbtrs_blocked: workspace of %zu bytes needed, %zu given", need, lwork);
        return BH_ERR_WORKSPACE;
    }
    int st = trs_blocked_prepare<T>(n, kl, ku, ab, ldab, ipiv, work, stream());
    if (st) return st;
    return trs_blocked_solve<T>(n, kl, ku, nrhs, ab, ldab, work, B, ldb, stream());
}

extern "C" {

int bh_gbtrs_blocked_workspace(char prec, bh_int n, bh_int kl, bh_int ku, size_t *bytes) {
    BH_ARG(prec == 'd' || prec == 's', 1);
    BH_ARG(n >= 0, 2);
    BH_ARG(kl >= 0, 3);
    BH_ARG(ku >= 0, 4);
    BH_ARG(bytes != nullptr, 5);
    *bytes = prec == 'd' ? trs_blocked_bytes<double>(n, kl, ku) : trs_blocked_bytes<float>(n, kl, ku);
    return BH_OK;
}

int bh_dgbtrs_blocked(bh_int n, bh_int kl, bh_int ku, bh_int nrhs, const double *AB, bh_int ldab, const bh_int *ipiv,
                      double *B, bh_int ldb, void *work, size_t lwork) {
    return gbtrs_blocked_impl<double>(n, kl, ku, nrhs, AB, ldab, ipiv, B, ldb, work, lwork);
}

int bh_sgbtrs_blocked(bh_int n, bh_int kl, bh_int ku, bh_int nrhs, const float *AB, bh_int ldab, const bh_int *ipiv,
                      float *B, bh_int ldb, void *work, size_t lwork) {
    return gbtrs_blocked_impl<float>(n, kl, ku, nrhs, AB, ldab, ipiv, B, ldb, work, lwork);
}

}  // extern "C"
