// q8_0_prompt.hpp -- the G-mode product for prompts (q8_0_prompt.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ane {

// Whether the operands (W even, below 2 GiB) and the launch fit the kernel.
bool prompt_eligible(uint32_t N, uint32_t nb, uint32_t T, const void* W);
// y[T x N] from activations already quantized in the form of k_q8_0_mmv
// (q8_0_mmv.hpp, quantize_bt): qxb[b][Tp][32] int8, dxb[b][Tp] fp32, Tp = ceil16(T).
// -1 when not eligible (nothing queued).
int prompt_mul_mat(uint32_t N, uint32_t nb, uint32_t T, const void* W, const void* qxb, const float* dxb, uint32_t Tp,
                   float* y, hipStream_t s);

}  // namespace ane
