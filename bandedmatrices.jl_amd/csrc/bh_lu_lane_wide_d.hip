// bh_lu_lane_wide_d.hip -- the one-wave LU for double, 9 to 15 subdiagonals.
#define BH_LANE_T double
#define BH_LANE_WIDE
#include "bh_lu_lane.hpp"
