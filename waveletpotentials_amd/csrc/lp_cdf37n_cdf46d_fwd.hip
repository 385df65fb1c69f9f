// Line-parallel kernels of the pair curl CDF3.7 'n' / divergence CDF4.6 'd', forward direction
// (see line_parallel.h).
#include "line_parallel.h"

namespace whhd {
template bool lp_launch<W_Cdf37N, W_Cdf46D, true>(int, int, lp::LpJobs&, int, int, hipStream_t);
}  // namespace whhd
