// The DP kernels in FP64 with per-clade power-of-two exponents.
#include "dp.hpp"

WHALE_DP_INSTANTIATE(double, true)
