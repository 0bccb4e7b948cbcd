// bh_gbqr_lane_s.hip -- the narrow-band QR kernels for float.
#define BH_QL_T float
#include "bh_gbqr_lane.hpp"
