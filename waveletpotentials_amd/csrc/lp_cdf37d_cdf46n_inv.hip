// Line-parallel kernels of the pair curl CDF3.7 'd' / divergence CDF4.6 'n', inverse direction
// (see line_parallel.h).
#include "line_parallel.h"

namespace whhd {
template bool lp_launch<W_Cdf37D, W_Cdf46N, false>(int, int, lp::LpJobs&, int, int, hipStream_t);
}  // namespace whhd
