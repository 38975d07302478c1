// rmode_mul_mat.hpp -- the many-token R-mode product (rmode_mul_mat.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ane {

// y[t][m] (T x N fp32) = the R-mode product of x row t (K fp32, rows
// contiguous, K a multiple of 32) with weight row m, Q4_0 (q4) or Q8_0.
// Bit-identical to one ane_hip_q4_0_gemv / ane_hip_q8_0_gemv per token.
// -1 (nothing queued) for a shape it does not take: no blocks, weights at an
// odd address, operands of 2 GiB or more, y overlapping x, a launch that does
// not fit, two or three tokens that the GEMVs serve faster.
int rmode_mul_mat(bool q4, uint32_t N, uint32_t K, uint32_t T, const float* x, const void* W, float* y,
                  hipStream_t s);
// Whether N x T outputs fit one launch.
bool rmode_launch_fits(uint32_t N, uint32_t T);

}  // namespace ane
