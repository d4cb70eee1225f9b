// The DP kernels in FP32 with per-clade power-of-two exponents.
#include "dp.hpp"

WHALE_DP_INSTANTIATE(float, true)
