// The low-rank decays exp(-exp(w tanh(p) + w0)) on the matrix cores, 32-bit factors as three bfloat16 operands: what the kernels
// that compute them share.
#pragma once
#include "common.h"

namespace sa {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

// tanh of eight numbers as three bfloat16 operands: its rounding, the rounding of what that leaves, and the rest (all 24 bits), so
// that three products into one sum are that of 32-bit factors.  tanh by the hardware's exponential: 1 - 2 / (e^(2x) + 1), and
// x (1 - x^2 / 3) where that cancels.
__device__ __forceinline__ void tanh_in_three(const float (&xs)[8], bf16x8& hi, bf16x8& mid, bf16x8& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float x = xs[j];
    const float y = 1.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * x) + 1.f);
    const float th = fabsf(x) < 0.02f ? x * fmaf(x * x, -1.f / 3.f, 1.f) : y;
    hi[j] = static_cast<__bf16>(th);
    const float rest = th - static_cast<float>(hi[j]);
    mid[j] = static_cast<__bf16>(rest);
    lo[j] = static_cast<__bf16>(rest - static_cast<float>(mid[j]));
  }
}

__device__ __forceinline__ floatx4 product_in_three(bf16x8 w, bf16x8 hi, bf16x8 mid, bf16x8 lo, floatx4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, hi, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, mid, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, lo, acc, 0, 0, 0);
}

}  // namespace sa
