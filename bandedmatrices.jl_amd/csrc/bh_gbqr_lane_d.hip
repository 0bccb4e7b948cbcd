// bh_gbqr_lane_d.hip -- the narrow-band QR kernels for double.
#define BH_QL_T double
#include "bh_gbqr_lane.hpp"
