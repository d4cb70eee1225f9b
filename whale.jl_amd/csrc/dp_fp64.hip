// The DP kernels in FP64, the reference's recursion.
#include "dp.hpp"

WHALE_DP_INSTANTIATE(double, false)
