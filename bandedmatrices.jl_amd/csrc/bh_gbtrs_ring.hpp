// bh_gbtrs_ring.hpp -- band LU solve 'N' and 'T' with one wave per right-hand
// side, the vector held in a lane ring (no per-step lane shifts).  The
// launchers are instantiated one per unit (bh_gbtrs_ring_{n,t}_{d,s}.hip) so
// the fully unrolled kernels compile in parallel.
#pragma once
//
// Restates LAPACK xGBTRS 'N' (ldiv!(::BandedLU, B), src/banded/linalg.jl:24-30)
// with its rounding, so results are bit-identical:
//   forward  (j = 0 .. n-2): swap b_j <-> b_p (p = ipiv_j - 1),
//            b_{j+t} = fma(l_{j+t,j}, -b_j, b_{j+t}), t = 1 .. min(kl, n-1-j);
//   backward (j = n-1 .. 0): x_j = b_j / u_jj (a true division),
//            b_{j-t} = fma(u_{j-t,j}, -x_j, b_{j-t}), t = 1 .. min(kl+ku, j).
//
// Layout: entry e of b lives in lane e mod 64 of a register that holds one
// 64-entry block.  The wave walks the steps block by block (64 steps,
// unrolled, so lane and register of every operand are compile-time); the
// registers rotate once per block (the finished block is stored, the block
// entering the window is loaded one block ahead).  The factor columns are
// read straight from AB into registers PFD steps ahead of their use -- a lone
// wave on its CU can afford PFD * (window registers) VGPRs, which is what
// hides the memory latency; the step itself is register-only.
//
// Cut systems (bh_cut.hpp): each of the two sweeps runs by blocks of 64-step
// groups, one wave per right-hand side and block, B -> Y -> Z; a block's
// window at its end must equal the next block's at its begin.
#include "bh_common.hpp"
#include "bh_cut.hpp"

namespace bh {

namespace {

// What a launch runs: both sweeps of the whole system in place, or (cut) one
// of them by blocks from `in` to `out`.
template <typename T>
struct RingWork {
    int sweeps;  // 1: the first, 2: the second, 3: both
    const T *in;
    T *out;
    i64 ldin, ldout;
    SweepCut<T> cut;
};

template <int K>
struct SC {
    static constexpr int value = K;
};
template <int N>
struct Unroll {
    template <class F>
    __device__ __forceinline__ static void run(F &&f) {
        Unroll<N - 1>::run(f);
        f(SC<N - 1>{});
    }
};
template <>
struct Unroll<0> {
    template <class F>
    __device__ __forceinline__ static void run(F &&) {}
};

__device__ __forceinline__ int mini(int a, int b) { return a < b ? a : b; }

constexpr int kRingWord3 = 0x00020000;  // word 3 of a raw buffer resource (gfx9 family)
// A byte offset past the end of any AB the ring kernel takes (those are under
// 2 GiB - 16 MiB), with room for +-64 * 5 entries either side.
constexpr int kRingPastEnd = 0x7f800000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t ring_rsrc(const void *p, i64 bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, kRingWord3);
}
__device__ __forceinline__ double ring_ld(__amdgpu_buffer_rsrc_t r, int off, double) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ float ring_ld(__amdgpu_buffer_rsrc_t r, int off, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ void ring_st(__amdgpu_buffer_rsrc_t r, int off, double v) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, off, 0, 0);
}
__device__ __forceinline__ void ring_st(__amdgpu_buffer_rsrc_t r, int off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
}
// NF = 1 + ceil(kl/64) forward registers, NB = 1 + ceil((kl+ku)/64) backward
// registers, PFD = prefetch distance in steps (divides 64).  The window
// registers are only ever indexed with compile-time indices (an interchange
// selects with uniform conditions and replaces single lanes), and all memory
// goes through buffer resources: a lane with nothing to load passes an
// offset past the end and reads 0, so no access sits in a branch.
template <typename T, int NF, int NB, int PFD>
__global__ void __launch_bounds__(64) gbtrs_n_ring(int n, int kl, int ku, const T *__restrict__ ab, i64 ld,
                                                   const i64 *__restrict__ ipiv, RingWork<T> wk) {
    static_assert(64 % PFD == 0, "prefetch distance divides the block");
    constexpr int SZ = (int)sizeof(T);
    const int lane = threadIdx.x, blk = blockIdx.y;
    const CutGeom cg = wk.cut.g;
    if (cg.p > 0 ? cut_closed(wk.cut.flags) : (wk.cut.flags && !cut_failed(wk.cut.flags))) return;
    const int kd = kl + ku;
    const __amdgpu_buffer_rsrc_t rab = ring_rsrc(ab, ld * (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rbi = ring_rsrc(wk.in + (i64)blockIdx.x * wk.ldin, (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rb = ring_rsrc(wk.out + (i64)blockIdx.x * wk.ldout, (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rip = ring_rsrc(ipiv, (i64)n * 8);
    auto bload = [&](int e) { return ring_ld(rbi, (e >= 0 && e < n) ? e * SZ : -1, T()); };
    // this launch's groups of a sweep of G, in the order they run: q0 .. q1-1,
    // its own from qown
    const bool cutting = cg.p > 0;
    const int q0 = cutting ? cg.start(blk) : 0, qown = cutting ? cg.own(blk) : 0;
    auto qend = [&](int G) { return cutting ? cg.end(blk) : G; };
    auto keep = [&](int which, auto &w) {
        constexpr int NR = sizeof(w) / sizeof(T);
        T *d = wk.cut.at(blk, which, 64 * NR);
#pragma unroll
        for (int r = 0; r < NR; ++r) d[64 * r + lane] = w[r];
    };
    const bool keep0 = cutting && blk > 0, keep1 = cutting && blk + 1 < cg.p;

    // ------------------------------------------------------------ forward: L and pivots
    if (kl > 0 && n > 1 && (wk.sweeps & 1)) {
        const int nsteps = n - 1;
        const int G = (nsteps + 63) >> 6, q1 = qend(G);
        T w[NF];  // w[r]: block g + r
#pragma unroll
        for (int r = 0; r < NF; ++r) w[r] = bload(64 * (q0 + r) + lane);
        T lp[PFD][NF];
        // multipliers of step j for window register r, lane = entry j + t
        // Lanes outside rows 1..lm load whatever the band storage holds there
        // (the update below is masked); only offsets off either end of AB
        // matter, and those read 0.  A step past the end gets a base offset
        // past the end of AB.
        auto fetch = [&](int slot, int j, int s, int ln) {
            const int base = j < nsteps ? (int)((i64)j * ld + kd) * SZ : kRingPastEnd;
#pragma unroll
            for (int r = 0; r < NF; ++r) lp[slot][r] = ring_ld(rab, base + (64 * r + ln - s) * SZ, T());
        };
        Unroll<PFD>::run([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            fetch(s, 64 * q0 + s, s, lane);
        });
        auto piv = [&](int e) { return (int)__builtin_amdgcn_raw_buffer_load_b32(rip, e < nsteps ? e * 8 : -1, 0, 0) - 1; };
        int pvc = piv(64 * q0 + lane);
        for (int g = q0; g < q1; ++g) {
            const int j0 = 64 * g;
            if (keep0 && g == qown) keep(0, w);
            // the lane index goes through an empty asm once per block, so the
            // per-step lane offsets are recomputed (one add) instead of being
            // hoisted out of the loop as 64 * NF live registers
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int pvn = piv(j0 + 64 + lane);
            const T bnext = bload(64 * (g + NF) + lane);
            Unroll<64>::run([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                constexpr int slot = s % PFD;
                const int j = j0 + s;
                if (j < nsteps) {
                    const int lm = mini(kl, n - 1 - j);
                    const int p = __builtin_amdgcn_readlane(pvc, s);
                    if (p != j) {
                        const int pos = s + (p - j);
                        const int rr = pos >> 6, pl = pos & 63;
                        T wsel = w[0];
#pragma unroll
                        for (int r = 1; r < NF; ++r)
                            if (rr == r) wsel = w[r];
                        const T bp = lane_read(wsel, pl);
                        const T bj0 = lane_read(w[0], s);
                        w[0] = lane_write(w[0], bp, s);
#pragma unroll
                        for (int r = 0; r < NF; ++r)
                            if (r == rr) w[r] = lane_write(w[r], bj0, pl);
                    }
                    const T nb = -lane_read(w[0], s);
#pragma unroll
                    for (int r = 0; r < NF; ++r) {
                        const int t = 64 * r + ln - s;
                        const T u = dfma(lp[slot][r], nb, w[r]);
                        w[r] = (t >= 1 && t <= lm) ? u : w[r];
                    }
                }
                fetch(slot, j + PFD, (s + PFD) & 63, ln);
            });
            ring_st(rb, (g >= qown && j0 + lane < n) ? (j0 + lane) * SZ : -1, w[0]);
#pragma unroll
            for (int r = 0; r + 1 < NF; ++r) w[r] = w[r + 1];
            w[NF - 1] = bnext;
            pvc = pvn;
        }
        if (keep1) keep(1, w);
#pragma unroll
        for (int r = 0; r < NF; ++r) {
            const int e = 64 * (G + r) + lane;
            ring_st(rb, (q1 == G && e < n) ? e * SZ : -1, w[r]);
        }
    }

    // the back substitution reads what the forward pass stored
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    // ------------------------------------------------------------ backward: U, kl+ku super-diagonals
    if (wk.sweeps & 2) {
        const int G = (n + 63) >> 6, q1 = qend(G), G0 = G - 1 - q0;
        T w[NB];  // w[r]: block g - r
#pragma unroll
        for (int r = 0; r < NB; ++r) w[r] = bload(64 * (G0 - r) + lane);
        T up[PFD][NB];
        // column j of U for window register r, lane = entry j - t (t = 0: diagonal)
        auto fetch = [&](int slot, int j, int s, int ln) {
            const int base = (j >= 0 && j < n) ? (int)((i64)j * ld + kd) * SZ : kRingPastEnd;
#pragma unroll
            for (int r = 0; r < NB; ++r) up[slot][r] = ring_ld(rab, base - (s - ln + 64 * r) * SZ, T());
        };
        Unroll<PFD>::run([&](auto sc) {
            constexpr int s = 63 - decltype(sc)::value;
            fetch(s % PFD, 64 * G0 + s, s, lane);
        });
        for (int q = q0; q < q1; ++q) {
            const int g = G - 1 - q, j0 = 64 * g;
            if (keep0 && q == qown) keep(0, w);
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const T bnext = bload(64 * (g - NB) + lane);
            Unroll<64>::run([&](auto sc) {
                constexpr int s = 63 - decltype(sc)::value;
                constexpr int slot = s % PFD;
                const int j = j0 + s;
                if (j <= n - 1) {
                    const T ujj = lane_read(up[slot][0], s);
                    const T xj = lane_read(w[0], s) / ujj;
                    w[0] = lane_write(w[0], xj, s);
                    const T nx = -xj;
                    const int tm = mini(kd, j);
#pragma unroll
                    for (int r = 0; r < NB; ++r) {
                        const int t = s - ln + 64 * r;
                        const T u = dfma(up[slot][r], nx, w[r]);
                        w[r] = (t >= 1 && t <= tm) ? u : w[r];
                    }
                }
                fetch(slot, j - PFD, (s - PFD) & 63, ln);
            });
            ring_st(rb, (q >= qown && j0 + lane < n) ? (j0 + lane) * SZ : -1, w[0]);
#pragma unroll
            for (int r = 0; r + 1 < NB; ++r) w[r] = w[r + 1];
            w[NB - 1] = bnext;
        }
        if (keep1) keep(1, w);
    }
}

// 'T' solve (transpose(F) \ B, src/banded/linalg.jl:41-47): U' y = b with
// j ascending, x_j = (b_j - sum_t u_{j-t,j} x_{j-t}) / u_jj, then L' with the
// interchanges in reverse, b_j -= sum_t l_{j+t,j} b_{j+t} followed by the swap
// b_j <-> b_{ipiv_j}.  Each step is a dot product over the band entries of
// one factor column (contiguous in band storage, so one coalesced load per
// window register) with the finished entries held in the lane ring, summed
// across the wave with DPP.  The dots are summed in a different order than
// the CPU routine's, so results agree to rounding, not bit for bit.
template <typename T, int NF, int NB, int PFD>
__global__ void __launch_bounds__(64) gbtrs_t_ring(int n, int kl, int ku, const T *__restrict__ ab, i64 ld,
                                                   const i64 *__restrict__ ipiv, RingWork<T> wk) {
    static_assert(64 % PFD == 0, "prefetch distance divides the block");
    constexpr int SZ = (int)sizeof(T);
    const int lane = threadIdx.x, blk = blockIdx.y;
    const CutGeom cg = wk.cut.g;
    if (cg.p > 0 ? cut_closed(wk.cut.flags) : (wk.cut.flags && !cut_failed(wk.cut.flags))) return;
    const int kd = kl + ku;
    const __amdgpu_buffer_rsrc_t rab = ring_rsrc(ab, ld * (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rbi = ring_rsrc(wk.in + (i64)blockIdx.x * wk.ldin, (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rb = ring_rsrc(wk.out + (i64)blockIdx.x * wk.ldout, (i64)n * SZ);
    const __amdgpu_buffer_rsrc_t rip = ring_rsrc(ipiv, (i64)n * 8);
    auto bload = [&](int e) { return ring_ld(rbi, (e >= 0 && e < n) ? e * SZ : -1, T()); };
    // this launch's groups of a sweep of G, in the order they run: q0 .. q1-1,
    // its own from qown
    const bool cutting = cg.p > 0;
    const int q0 = cutting ? cg.start(blk) : 0, qown = cutting ? cg.own(blk) : 0;
    auto qend = [&](int G) { return cutting ? cg.end(blk) : G; };
    auto keep = [&](int which, auto &w) {
        constexpr int NR = sizeof(w) / sizeof(T);
        T *d = wk.cut.at(blk, which, 64 * NR);
#pragma unroll
        for (int r = 0; r < NR; ++r) d[64 * r + lane] = w[r];
    };
    const bool keep0 = cutting && blk > 0, keep1 = cutting && blk + 1 < cg.p;

    // ------------------------------------------------------------ U' (ascending)
    if (wk.sweeps & 1) {
        const int G = (n + 63) >> 6, q1 = qend(G);
        T P[NB];  // P[r]: block g - r; entries below j are finished (none yet)
        P[0] = bload(64 * q0 + lane);
#pragma unroll
        for (int r = 1; r < NB; ++r) P[r] = T(0);
        T up[PFD][NB];
        // column j of U: lane L of register r holds u_{64(g-r)+L, j}, at t = s - L + 64r above the diagonal
        auto fetch = [&](int slot, int j, int s, int ln) {
            const int base = j < n ? (int)((i64)j * ld + kd) * SZ : kRingPastEnd;
#pragma unroll
            for (int r = 0; r < NB; ++r) up[slot][r] = ring_ld(rab, base - (s - ln + 64 * r) * SZ, T());
        };
        Unroll<PFD>::run([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            fetch(s, 64 * q0 + s, s, lane);
        });
        for (int g = q0; g < q1; ++g) {
            const int j0 = 64 * g;
            if (keep0 && g == qown) keep(0, P);
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const T bnext = bload(64 * (g + 1) + lane);
            Unroll<64>::run([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                constexpr int slot = s % PFD;
                const int j = j0 + s;
                if (j < n) {
                    const int tm = mini(kd, j);
                    T part = T(0);
#pragma unroll
                    for (int r = 0; r < NB; ++r) {
                        const int t = s - ln + 64 * r;
                        const T q = dfma(up[slot][r], P[r], part);
                        part = (t >= 1 && t <= tm) ? q : part;
                    }
                    const T dot = wave_sum_dpp(part);
                    const T xj = (lane_read(P[0], s) - dot) / lane_read(up[slot][0], s);
                    P[0] = lane_write(P[0], xj, s);
                }
                fetch(slot, j + PFD, (s + PFD) & 63, ln);
            });
            ring_st(rb, (g >= qown && j0 + lane < n) ? (j0 + lane) * SZ : -1, P[0]);
#pragma unroll
            for (int r = NB - 1; r >= 1; --r) P[r] = P[r - 1];
            P[0] = bnext;
        }
        if (keep1) keep(1, P);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    // ------------------------------------------------------------ L' and the interchanges (descending)
    if (kl > 0 && n > 1 && (wk.sweeps & 2)) {
        const int G = ((n - 2) >> 6) + 1, q1 = qend(G), g0 = G - 1 - q0;
        T F[NF];  // F[r]: block g + r; entries above j are finished
        // (row n-1 is from the start; a later block begins with none)
#pragma unroll
        for (int r = 0; r < NF; ++r) F[r] = (r == 0 || q0 == 0) ? bload(64 * (g0 + r) + lane) : T(0);
        T lp[PFD][NF];
        // column j of L: lane L of register r holds l_{64(g+r)+L, j}, at t = 64r + L - s below the diagonal
        auto fetch = [&](int slot, int j, int s, int ln) {
            const int base = (j >= 0 && j < n - 1) ? (int)((i64)j * ld + kd) * SZ : kRingPastEnd;
#pragma unroll
            for (int r = 0; r < NF; ++r) lp[slot][r] = ring_ld(rab, base + (64 * r + ln - s) * SZ, T());
        };
        Unroll<PFD>::run([&](auto sc) {
            constexpr int s = 63 - decltype(sc)::value;
            fetch(s % PFD, 64 * g0 + s, s, lane);
        });
        auto piv = [&](int e) {
            return (int)__builtin_amdgcn_raw_buffer_load_b32(rip, (e >= 0 && e < n - 1) ? e * 8 : -1, 0, 0) - 1;
        };
        for (int q = q0; q < q1; ++q) {
            const int g = G - 1 - q, j0 = 64 * g;
            if (keep0 && q == qown) keep(0, F);
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int pvb = piv(j0 + lane);
            const T bprev = bload(64 * (g - 1) + lane);
            Unroll<64>::run([&](auto sc) {
                constexpr int s = 63 - decltype(sc)::value;
                constexpr int slot = s % PFD;
                const int j = j0 + s;
                if (j <= n - 2) {
                    const int lm = mini(kl, n - 1 - j);
                    T part = T(0);
#pragma unroll
                    for (int r = 0; r < NF; ++r) {
                        const int t = 64 * r + ln - s;
                        const T q = dfma(lp[slot][r], F[r], part);
                        part = (t >= 1 && t <= lm) ? q : part;
                    }
                    const T dot = wave_sum_dpp(part);
                    T bj = lane_read(F[0], s) - dot;
                    const int p = __builtin_amdgcn_readlane(pvb, s);
                    if (p != j) {
                        const int pos = s + (p - j);
                        const int rr = pos >> 6, pl = pos & 63;
                        T fsel = F[0];
#pragma unroll
                        for (int r = 1; r < NF; ++r)
                            if (rr == r) fsel = F[r];
                        const T bp = lane_read(fsel, pl);
#pragma unroll
                        for (int r = 0; r < NF; ++r)
                            if (r == rr) F[r] = lane_write(F[r], bj, pl);
                        bj = bp;
                    }
                    F[0] = lane_write(F[0], bj, s);
                }
                fetch(slot, j - PFD, (s - PFD) & 63, ln);
            });
            // the top block is finished: no later step reaches it
            const int et = 64 * (g + NF - 1) + lane;
            ring_st(rb, (q >= qown && et < n) ? et * SZ : -1, F[NF - 1]);
#pragma unroll
            for (int r = NF - 1; r >= 1; --r) F[r] = F[r - 1];
            F[0] = bprev;
        }
        if (keep1) keep(1, F);
#pragma unroll
        for (int r = 1; r < NF; ++r) {
            const int e = 64 * (r - 1) + lane;
            ring_st(rb, (q1 == G && e < n) ? e * SZ : -1, F[r]);
        }
    }
}

}  // namespace

// Both sweeps with one kernel.  `how`: 0 the whole system; 1 by blocks if it
// can be cut, and behind them the whole system, which does nothing where they
// agreed; for a caller with another fallback, that waits for the verdicts: 2
// the gate alone (*cw: the memory, or none), 3 the blocks behind it.  Gate: U's
// columns at 1.25 times the rest of the column, L's multipliers summing to less
// than 0.8.  Measured FP64 1 RHS against the whole sweeps: n = 262144, (16,16)
// the two solves of a gradient 5.3 -> 0.7 ms (60.7 and 100 ms as whole sweeps,
// 2.6 and 2.7 partitioned).
template <typename T, int NF, int NB, class K>
int ring_run(K kern, bool trans, int how, i64 n, i64 kl, i64 ku, i64 nrhs, const T *ab, i64 ld, const i64 *ipiv, T *B,
             i64 ldb, hipStream_t st, RingCutWs *cw) {
    const dim3 block(64);
    const i64 kd = kl + ku;
    RingWork<T> seq{3, B, B, ldb, ldb, SweepCut<T>{}};
    // the sweep with L has n-1 steps, the one with U n
    const CutGeom gu = sweep_geom<T>(n, kd, nrhs, NB), gl = sweep_geom<T>(n - 1, kl, nrhs, NF);
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t by = al((size_t)n * nrhs * sizeof(T));
    const size_t su = al((size_t)gu.p * nrhs * 2 * 64 * NB * sizeof(T));
    const size_t sl = kl ? al((size_t)gl.p * nrhs * 2 * 64 * NF * sizeof(T)) : 0;
    char *ws = how == 3 ? (char *)cw->ws : nullptr;
    int *flags = how == 3 ? cw->flags : nullptr, *host = how == 3 ? cw->host : nullptr;
    if (how == 1 || how == 2) cut_begin();
    if ((how == 1 || how == 2) && gu.p > 0 && (kl == 0 || gl.p > 0) && cut_enabled()) {
        if (how == 2) host = cut_host_words();
        if (how == 1 || host) ws = (char *)cut_alloc(2 * by + su + sl + 256, st);
        if (ws) {
            flags = (int *)(ws + 2 * by + su + sl);
            hipLaunchKernelGGL(cut_gate<T>, dim3(1), dim3(1024), 0, st, ab, ld, (int)n,
                               CutSet{0, (int)kd + 1, (int)kd, 0}, CutSet{(int)kd, kl ? (int)kl + 1 : 0, (int)kd, 1},
                               5, 0.0f, flags, host, (i64 *)nullptr);
            cut_note(flags, st);
        }
    }
    if (ws && how != 2) {
        T *Y = (T *)ws, *Z = (T *)(ws + by), *snu = (T *)(ws + 2 * by), *snl = (T *)(ws + 2 * by + su);
        const T *in = B;
        i64 ldin = ldb;
        T *out = Y;
        for (int sweep = 1; sweep <= 2; ++sweep) {
            const bool lower = trans == (sweep == 2);
            if (lower && kl == 0) continue;
            const CutGeom &g = lower ? gl : gu;
            T *snap = lower ? snl : snu;
            hipLaunchKernelGGL(kern, dim3((unsigned)nrhs, g.p), block, 0, st, (int)n, (int)kl, (int)ku, ab, ld, ipiv,
                               RingWork<T>{sweep, in, out, ldin, n, SweepCut<T>{g, flags, snap}});
            hipLaunchKernelGGL(sweep_check<T>, dim3(g.p - 1, (unsigned)nrhs), dim3(256), 0, st, (const T *)snap,
                               64 * (lower ? NF : NB), flags);
            in = out;
            ldin = n;
            out = Z;
        }
        hipLaunchKernelGGL(sweep_commit<T>, dim3((unsigned)cdiv(n, 256), (unsigned)nrhs), dim3(256), 0, st, (int)n, in,
                           B, 1, ldb, (const int *)flags, host ? host + 1 : nullptr);
        seq.cut.flags = flags;
    }
    if (how < 2)
        hipLaunchKernelGGL(kern, dim3((unsigned)nrhs), block, 0, st, (int)n, (int)kl, (int)ku, ab, ld, ipiv, seq);
    const hipError_t e = hipGetLastError();
    if (how < 2 || (how == 2 && e != hipSuccess)) {
        cut_free(ws, st);
        ws = nullptr;
    }
    if (how == 2) *cw = RingCutWs{ws, flags, host};
    return e == hipSuccess ? BH_OK : hip_fail(e, "kernel launch", __FILE__, __LINE__);
}

// The solve for bands with kl <= 128 and kl + ku <= 256; -1 otherwise.
#define BH_RING_LAUNCH(NAME, KERN, TRANS)                                                                            \
    template <typename T>                                                                                            \
    int NAME(int how, i64 n, i64 kl, i64 ku, i64 nrhs, const T *ab, i64 ld, const i64 *ipiv, T *B, i64 ldb,          \
             hipStream_t st, RingCutWs *cw) {                                                                        \
        const i64 kd = kl + ku;                                                                                      \
        if (n >= (1ll << 30) || kl > 128 || kd > 256 || ld * n * (i64)sizeof(T) >= (1ll << 31) - (1ll << 24))        \
            return -1;                                                                                               \
        const int nf = 1 + (int)cdiv(kl, 64), nb = 1 + (int)cdiv(kd, 64);                                            \
        constexpr int PFD = sizeof(T) == 4 ? 32 : 16;                                                                \
        if (nf <= 2 && nb <= 2)                                                                                      \
            return ring_run<T, 2, 2>(KERN<T, 2, 2, PFD>, TRANS, how, n, kl, ku, nrhs, ab, ld, ipiv, B, ldb, st, cw); \
        if (nf <= 2 && nb <= 3)                                                                                      \
            return ring_run<T, 2, 3>(KERN<T, 2, 3, PFD>, TRANS, how, n, kl, ku, nrhs, ab, ld, ipiv, B, ldb, st, cw); \
        if (nf <= 3 && nb <= 3)                                                                                      \
            return ring_run<T, 3, 3>(KERN<T, 3, 3, PFD>, TRANS, how, n, kl, ku, nrhs, ab, ld, ipiv, B, ldb, st, cw); \
        return ring_run<T, 3, 5>(KERN<T, 3, 5, PFD>, TRANS, how, n, kl, ku, nrhs, ab, ld, ipiv, B, ldb, st, cw);     \
    }
#if BH_RING_TRANS
BH_RING_LAUNCH(ring_gbtrs_t_launch, gbtrs_t_ring, true)
#else
BH_RING_LAUNCH(ring_gbtrs_launch, gbtrs_n_ring, false)
#endif
#undef BH_RING_LAUNCH

}  // namespace bh
