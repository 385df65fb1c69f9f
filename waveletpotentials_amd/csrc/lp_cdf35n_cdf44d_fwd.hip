// Line-parallel kernels of the pair curl CDF3.5 'n' / divergence CDF4.4 'd', forward direction
// (see line_parallel.h).
#include "line_parallel.h"

namespace whhd {
template bool lp_launch<W_Cdf35N, W_Cdf44D, true>(int, int, lp::LpJobs&, int, int, hipStream_t);
}  // namespace whhd
