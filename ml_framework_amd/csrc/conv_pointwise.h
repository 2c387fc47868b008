// conv_pointwise.h -- 1x1 stride-1 convolutions in one pass over memory
// (conv_pointwise.hip). Each reports in *used whether it ran (false: sizes or
// addresses out of its range, or no scratch to be had).
#pragma once

#include <hip/hip_runtime.h>

#include "conv_band.h"

namespace seera {

// Y [B, F, HW] = act(Wt [F, C] . X [B, C, HW] + bias).
int pointwise_conv_fwd(const float* X, const float* Wt, float* Y, int B, int C, int64_t HW, int F, const ConvEpi& epi,
                       hipStream_t st, bool* used);

// dX, dW and (db not nullptr) db of the same layer.
int pointwise_conv_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW, float* db, int B, int C,
                       int64_t HW, int F, hipStream_t st, bool* used);

}  // namespace seera
