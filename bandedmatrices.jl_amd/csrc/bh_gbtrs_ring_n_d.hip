// bh_gbtrs_ring_n_d.hip -- the FP64 'N' lane-ring band solve (kernels in
// bh_gbtrs_ring.hpp), a unit of its own so the ring kernels compile in parallel.
#define BH_RING_TRANS 0
#include "bh_gbtrs_ring.hpp"

namespace bh {
template int ring_gbtrs_launch<double>(int, i64, i64, i64, i64, const double *, i64, const i64 *, double *, i64,
                                   hipStream_t, RingCutWs *);
}  // namespace bh
