// What the recurrences that take a prompt's tokens in pieces of 64 on the f32 matrix instructions have in common
// (delta_chunks.hip, linear_chunks.hip).  A 16 x 16 result holds rows 4 g + r (g = lane / 16, r = 0 .. 3) and column
// c = lane % 16; of the four steps over 16 entries of the sum, step r takes entries 4 g + r of both operands.
#pragma once
#include "attention_common.h"

namespace sa {
namespace chunks {

constexpr int kTokens = 64, kBlocks = kTokens / 16;
constexpr int kBlock = 256;   // floats of a 16 x 16 block

struct Span {
  int slot, first, count, piece0;
};
// The part of request `seq` that lies in rows row0 .. row1 - 1 of the step; its pieces are numbered from piece0 on, no two
// requests' alike.
__device__ __forceinline__ Span span_of(const int* seq_meta, int row0, int row1, int seq) {
  const int* meta = seq_meta + 4 * seq;
  const int lo = meta[1] > row0 ? meta[1] : row0, end = meta[1] + meta[2], hi = end < row1 ? end : row1;
  Span s;
  s.slot = meta[0];
  s.first = lo;
  s.count = hi - lo;
  s.piece0 = (lo - row0) / kTokens + seq;
  return s;
}

__device__ __forceinline__ floatx4 mul4(floatx4 a, floatx4 b, floatx4 c) {   // four steps: 16 channels or tokens
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}

// a . b alone, the four steps' sums by halves: a chain rounds at the size of the sum so far with every product, whose order it
// cannot choose.
__device__ __forceinline__ floatx4 halves4(floatx4 a, floatx4 b) {
  floatx4 x[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) x[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  return (x[0] + x[1]) + (x[2] + x[3]);
}

// The chains' sums, by halves.
template <int N>
__device__ __forceinline__ floatx4 sum_of(floatx4 (&x)[N]) {
#pragma unroll
  for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i) x[i] += x[i + n];
  return x[0];
}

// acc + m . b for a lower triangular m: the diagonal block of a product over earlier tokens.  A product with a zero carries an
// entry of b that is not finite into every row; such entries are left out of the product, and added one at a time to the rows
// at and behind their own.  IN_TIME: step r of the operands holds tokens 4 r + g instead of 4 g + r.
template <bool IN_TIME>
__device__ __forceinline__ floatx4 lower_mul4(floatx4 m, floatx4 b, floatx4 acc, int lane) {
  bool odd = false;
#pragma unroll
  for (int r = 0; r < 4; ++r) odd |= !(fabsf(b[r]) < INFINITY);
  if (__builtin_amdgcn_ballot_w64(odd) == 0) return mul4(m, b, acc);
  const int g = lane / 16;
  floatx4 finite;
#pragma unroll
  for (int r = 0; r < 4; ++r) finite[r] = fabsf(b[r]) < INFINITY ? b[r] : 0.f;
  acc = mul4(m, finite, acc);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll 1
    for (int of = 0; of < 4; ++of) {   // entry 4 of + r, or 4 r + of
      const bool mine = of == g && !(fabsf(b[r]) < INFINITY);
      if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
      const floatx4 one = __builtin_amdgcn_mfma_f32_16x16x4f32(of == g ? m[r] : 0.f, mine ? b[r] : 0.f,
                                                               floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += 4 * g + i >= (IN_TIME ? 4 * r + of : 4 * of + r) ? one[i] : 0.f;
    }
  }
  return acc;
}

}  // namespace chunks
}  // namespace sa
