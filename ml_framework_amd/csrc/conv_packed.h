// conv_packed.h -- host entry points of the packed-operand convolution path
// (conv_packed.hip). Each reports in *used whether it ran (false: sizes out of
// its range, or no staging memory to be had), and leaves the call to the other
// paths if not.
#pragma once

#include <hip/hip_runtime.h>

#include "conv_band.h"

namespace seera {

// Y = act(conv(X, Wt) + bias).
int packed_conv_fwd(const float* X, const float* Wt, float* Y, int B, int C, int H, int W, int F,
                    int R, int S, int sh, int sw, int ph, int pw, const ConvEpi& epi,
                    hipStream_t st, bool* used);

// dX, dW and (db not nullptr) db of the same layer.
int packed_conv_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW,
                    float* db, int B, int C, int H, int W, int F, int R, int S, int sh, int sw,
                    int ph, int pw, hipStream_t st, bool* used);

// Transposed convolution of X [B, F, Hi, Wi] to out [B, C, H, W] (Wt [F, C, R,
// S]), and its gradients.
int packed_convT_fwd(const float* X, const float* Wt, float* out, int B, int F, int Hi, int Wi, int C,
                     int H, int W, int R, int S, int sh, int sw, int ph, int pw, hipStream_t st,
                     bool* used);
int packed_convT_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW, int B,
                     int F, int Hi, int Wi, int C, int H, int W, int R, int S, int sh, int sw, int ph,
                     int pw, hipStream_t st, bool* used);

// The first two for a first layer (stride 2, kernel 7 or 8 wide, at most 4
// channels) in space-to-depth form.
int packed_stem_fwd(const float* X, const float* Wt, float* Y, int B, int C, int H, int W, int F,
                    int R, int S, int sh, int sw, int ph, int pw, const ConvEpi& epi,
                    hipStream_t st, bool* used);
int packed_stem_bwd(const float* dY, const float* Wt, const float* X, float* dX, float* dW, float* db,
                    int B, int C, int H, int W, int F, int R, int S, int sh, int sw, int ph, int pw,
                    hipStream_t st, bool* used);

}  // namespace seera
