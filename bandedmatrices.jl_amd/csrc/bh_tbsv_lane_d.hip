// bh_tbsv_lane_d.hip -- the one-lane-per-block triangular solve for double.
#define BH_TL_T double
#include "bh_tbsv_lane.hpp"

namespace bh {

// Lead-in as sweep_geom's (20 k steps in FP64, 10 k in FP32, and the window);
// up to 16384 lanes (one wave to a CU) and at least 32 own steps.
TbsvLane tbsv_lane_geom(i64 n, i64 k, i64 lda, i64 incx, i64 ldx, i64 nrhs, int elem) {
    TbsvLane g;
    const i64 lim = (1ll << 31) - (1 << 24);
    if (k < 1 || k > 16 || nrhs > 1024 || n >= (1ll << 29) || lda * n * elem >= lim || n * incx * elem >= lim) return g;
    const i64 R = k <= 7 ? 8 : k <= 10 ? k + 1 : (k + 2) / 2 * 2;
    const i64 W = R * cdiv((elem == 8 ? 20 : 10) * k + 32, R);
    const i64 L = R * cdiv(imax(32, cdiv(n * nrhs, 16384)), R);
    if (3 * (L + W) > n) return g;
    g.L = (int)L;
    g.W = (int)W;
    g.p = (int)cdiv(n, L);
    return g;
}

}  // namespace bh
