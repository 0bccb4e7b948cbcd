// bh_lu_lane_wide_s.hip -- the one-wave LU for float, 9 to 15 subdiagonals.
#define BH_LANE_T float
#define BH_LANE_WIDE
#include "bh_lu_lane.hpp"
