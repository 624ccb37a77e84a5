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

// Whether the states in front of the pieces are kept and the outputs made from them afterwards (piece_outputs_kernel), instead of by
// the walk: where the walk is long and leaves half of the CUs idle.  What is kept goes through memory, which costs more than it
// gives with more walkers.  Delta rule and decays per channel, heads of 128, us (walk with outputs / kept):
//   16 heads, tokens       256: 41 / 50, 44 / 50   512: 60 / 65, 55 / 56   1,024: 85 / 82, 78 / 66   2,048: 137 / 121, 126 / 91
//   8 heads                512: 52 / 56, 53 / 52   2,048: 131 / 105, 114 / 72
//   32 heads               2,048: 181 / 217, 165 / 167
constexpr bool keeps_states(int longest, int64_t walkers) { return longest >= 768 && walkers <= 128; }

// Where the outputs of a piece find their operands, floats behind the piece's first: scaled queries and weights of tokens as left
// operands, [token block][channel block] and [token block][token block], what tokens add as right operands [column block][token
// block], the state in front of the piece [column block][channel block], and (OWN) what the tokens' own weights are.
struct OutputsAt {
  int q, p, v, states, own, words;
};

// out = q S + p v for all pieces of 64 tokens at once, a workgroup per piece and head: with the states in front of the pieces kept by
// the walk, outputs are no part of its chain.  Queries and weights lie in LDS for the four waves, each of which takes every fourth
// block of 16 value columns.  The sums are the walk's, in the same order.  OWN: the diagonal of p by itself; else p holds it and the
// tokens are IN_TIME.  2,048 tokens of 16 heads of 128: 28 and 25 us, 74 MB and 340 matrix instructions a wave, one after the other.
template <int NT, bool OWN>
__global__ __launch_bounds__(256, 2) void piece_outputs_kernel(const float* __restrict__ pieces, OutputsAt at, const int* __restrict__ seq_meta,
                                                            int row0, int row1, int H, int dv, float* __restrict__ out) {
  __shared__ __align__(16) float q_s[kBlocks * NT * kBlock], p_s[kBlocks * kBlocks * kBlock];
  const Span sp = span_of(seq_meta, row0, row1, blockIdx.z);
  const int t0 = blockIdx.y * kTokens;
  if (t0 >= sp.count) return;   // (uniform)
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), c = lane % 16, g = lane / 16;
  const float* piece = pieces + (static_cast<size_t>(sp.piece0 + blockIdx.y) * H + h) * at.words;
  const int cb = (dv + 15) / 16;
  floatx4 st[NT], v[kBlocks];
  auto fetch = [&](int n) __attribute__((always_inline)) {   // column block n (behind the last: that one, not used)
    const int j = n < cb ? n : cb - 1;
#pragma unroll
    for (int i = 0; i < NT; ++i) st[i] = *reinterpret_cast<const floatx4*>(piece + at.states + (j * NT + i) * kBlock + lane * 4);
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) v[b] = *reinterpret_cast<const floatx4*>(piece + at.v + (j * kBlocks + b) * kBlock + lane * 4);
  };
  fetch(wave);
#pragma unroll
  for (int i = 0; i < kBlocks * NT / 4; ++i)
    reinterpret_cast<floatx4*>(q_s)[tid + i * 256] = *reinterpret_cast<const floatx4*>(piece + at.q + (tid + i * 256) * 4);
#pragma unroll
  for (int i = 0; i < kBlocks; ++i) {   // (token block i; blocks behind the diagonal are not there, and not used)
    const int b = wave < i ? wave : i;
    reinterpret_cast<floatx4*>(p_s)[tid + i * 256] = *reinterpret_cast<const floatx4*>(piece + at.p + (i * kBlocks + b) * kBlock + lane * 4);
  }
  __syncthreads();
  for (int n = wave; n < cb; n += 4) {
    const int col = n * 16 + c;
#pragma unroll 1
    for (int t = 0; t < kBlocks; ++t) {   // (one at a time: four at once take more registers than two waves of a SIMD have)
      const floatx4 v_own = t == 0 ? v[0] : t == 1 ? v[1] : t == 2 ? v[2] : v[3];
      constexpr int CHAINS = OWN ? 4 : NT;
      floatx4 o[CHAINS], o2[kBlocks];
#pragma unroll
      for (int i = 0; i < CHAINS; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NT; ++i)
        o[i % CHAINS] = mul4(reinterpret_cast<const floatx4*>(q_s)[(t * NT + i) * kWave + lane], st[i], o[i % CHAINS]);
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) o2[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < kBlocks - 1; ++b)
        if (b < t) o2[b] = mul4(reinterpret_cast<const floatx4*>(p_s)[(t * kBlocks + b) * kWave + lane], v[b], o2[b]);
      o2[kBlocks - 1] = lower_mul4<!OWN>(reinterpret_cast<const floatx4*>(p_s)[(t * kBlocks + t) * kWave + lane], v_own, o2[kBlocks - 1], lane);
      floatx4 result = sum_of(o) + sum_of(o2);
      if (OWN) {
        const floatx4 own = *reinterpret_cast<const floatx4*>(piece + at.own + t * 16 + g * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) result[r] = fmaf(own[r], v_own[r], result[r]);
      }
      if (col < dv) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = t0 + t * 16 + g * 4 + r;
          if (i < sp.count) out[static_cast<size_t>(sp.first + i) * (static_cast<size_t>(H) * dv) + static_cast<size_t>(h) * dv + col] = result[r];
        }
      }
    }
    fetch(n + 4);
  }
}

}  // namespace chunks
}  // namespace sa
