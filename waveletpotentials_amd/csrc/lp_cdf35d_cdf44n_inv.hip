// Line-parallel kernels of the pair curl CDF3.5 'd' / divergence CDF4.4 'n', inverse direction
// (see line_parallel.h).
#include "line_parallel.h"

namespace whhd {
template bool lp_launch<W_Cdf35D, W_Cdf44N, false>(int, int, lp::LpJobs&, int, int, hipStream_t);
}  // namespace whhd
