// Eight neighbouring entries of a row: one load or store of 16 bytes (bfloat16) or two (32-bit), widened to 32 bits.
#pragma once
#include "common.h"

namespace sa {

struct Eight {
  float v[8];
};
__device__ __forceinline__ Eight load_eight(const float* p) {
  Eight e;
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  e.v[0] = a.x, e.v[1] = a.y, e.v[2] = a.z, e.v[3] = a.w, e.v[4] = b.x, e.v[5] = b.y, e.v[6] = b.z, e.v[7] = b.w;
  return e;
}
__device__ __forceinline__ Eight load_eight(const bf16* p) {
  Eight e;
  const uint4 a = *reinterpret_cast<const uint4*>(p);
  const uint32_t u[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    e.v[2 * i] = __uint_as_float(u[i] << 16);
    e.v[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
  }
  return e;
}
__device__ __forceinline__ void store_eight(float* p, const Eight& e) {
  reinterpret_cast<float4*>(p)[0] = float4{e.v[0], e.v[1], e.v[2], e.v[3]};
  reinterpret_cast<float4*>(p)[1] = float4{e.v[4], e.v[5], e.v[6], e.v[7]};
}
__device__ __forceinline__ void store_eight(bf16* p, const Eight& e) {
  uint32_t u[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    u[i] = static_cast<uint32_t>(float_to_bf16(e.v[2 * i]).bits) | (static_cast<uint32_t>(float_to_bf16(e.v[2 * i + 1]).bits) << 16);
  *reinterpret_cast<uint4*>(p) = uint4{u[0], u[1], u[2], u[3]};
}

}  // namespace sa
