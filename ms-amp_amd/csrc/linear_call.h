// What the calls for a linear layer's directions use of the cast kernels.
#pragma once

#include "common.cuh"

namespace msamp {

// The casts of a linear layer's forward (x and the weight), of its backward (dy, with the column sums into bias_sum if it is given
// and the old weight gradient, if there is one, dequantized into `product`) ...
int cast_linear_inputs(const msamp_linear_forward_args& a, hipStream_t st);
int cast_output_gradient(const msamp_linear_backward_args& a, void* product, float* sums, hipStream_t st);
// ... and of a forward of a few tokens:
// x[tokens][K] (K a multiple of 16) to E4M3 as msamp_cast_to_fp8_gated casts it, the codes in the order in which the product of a
// few tokens reads them: for every 128-wide slice of K, block of 16 tokens and half slice 64 lanes of 16 bytes, lane l those of token
// l % 16 and k = 16 * (l / 16) .. +15 of the half; zeros past the last token and the last k.
int few_cast_fragments(const void* x, int in_dtype, int tokens, int K, float* scale, float* amax, float* scale_inv, uint8_t* out,
                       int flags, const int32_t* counter, int window, void* workspace, hipStream_t st);

}    // namespace msamp
