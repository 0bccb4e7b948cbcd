// bh_tbsv_lane_s.hip -- the one-lane-per-block triangular solve for float.
#define BH_TL_T float
#include "bh_tbsv_lane.hpp"
