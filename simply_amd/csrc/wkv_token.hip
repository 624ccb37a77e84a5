// A token of the matrix-state recurrence with low-rank decays and a bonus, with what stands around it, in one kernel:
//
//   a = exp(-exp(W tanh(p) + w0)),   o = (S + diag(u) k v^T)^T q,   S <- diag(a) S + k v^T,
//   out = o / sqrt(mean(o^2) + eps) * w * silu(g)      per head
//
// For decode steps: three launches in a row (the decays 5.2 us, the recurrence 13.1, norm and gate 4.8, at 8 requests of 16 heads
// of 128) that each wait for the one before become one of 9.8.  A workgroup of 8 waves takes one head of one request:
// its 64 KiB of state are asked for before anything else, whole columns of 16-byte pieces, and stay in registers while the decays
// (a wave a tile of 16 channels, on the matrix cores), the token's rows and the sums over a column's lanes are done; 128
// workgroups read and write 17 MB, 3 us at what HBM gives.  (The kernel for portions, linear_state_kernel, stages 16 tokens'
// operands in LDS for 8 columns at a time, which is what one token spent its time on.)
// Decays, sums, state and norm are 32-bit; a request's tokens go one after the other, in the same order of sums for any batch.
#include "api.h"
#include "common.h"
#include "low_rank.h"

namespace sa {

struct Four {
  float v[4];
};
__device__ __forceinline__ Four load_four(const bf16* p) {
  const uint2 q = *reinterpret_cast<const uint2*>(p);
  return Four{{__uint_as_float(q.x << 16), __uint_as_float(q.x & 0xffff0000u), __uint_as_float(q.y << 16),
               __uint_as_float(q.y & 0xffff0000u)}};
}

struct WkvToken {
  const bf16* proj;
  int64_t proj_stride;
  int q_at, k_at, v_at, g_at, low_at, rank;
  const bf16* decay_w;   // operand tiles [H * D / 16][rank / 32][64][8]
  const void *base, *bonus, *norm;
  int base_dtype, bonus_dtype, norm_dtype;
  float eps;
  int H;
  float* state;
  int64_t state_stride;
  const int* seq_meta;
  bf16* out;
};

constexpr int kTokenWaves = 8, kTokenChunks = 4;   // ranks of up to 128
template <int D>
__global__ __launch_bounds__(kTokenWaves * kWave) void wkv_token_kernel(WkvToken a) {
  constexpr int LPC = D / 4, PER = kWave / LPC;              // lanes of a column, columns of a load
  constexpr int LOADS = D / (kTokenWaves * PER);             // loads of a lane: 8 (heads of 128) or 2 (64)
  __shared__ float vs[D], os[D];
  __shared__ __align__(16) float decay_s[D];
  const int* meta = a.seq_meta + 4 * blockIdx.x;
  const int slot = meta[0], first = meta[1], count = meta[2];
  const int h = blockIdx.y, tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  if (count <= 0) return;   // (uniform)
  const int row = (lane % LPC) * 4, col0 = wave * LOADS * PER + lane / LPC;
  float* S = a.state + static_cast<size_t>(slot) * a.state_stride + static_cast<size_t>(h) * D * D + row;
  const int r16 = lane % 16, kq = lane / 16, chunks = (a.rank + 31) / 32;
  const bool decays = wave < D / 16;   // (a wave a tile of 16 channels)
  const bf16* tile = a.decay_w + (static_cast<size_t>(h) * (D / 16) + (decays ? wave : 0)) * chunks * 512 + lane * 8;
  bf16x8 wv[kTokenChunks];
#pragma unroll
  for (int c = 0; c < kTokenChunks; ++c)
    wv[c] = *reinterpret_cast<const bf16x8*>(tile + static_cast<size_t>(c < chunks ? c : chunks - 1) * 512);
  float bonus[4], base[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bonus[i] = load_f(a.bonus, a.bonus_dtype, static_cast<size_t>(h) * D + row + i);
    base[i] = load_f(a.base, a.base_dtype, static_cast<size_t>(h) * D + (decays ? wave * 16 : 0) + kq * 4 + i);
  }
  const float weight = tid < D ? load_f(a.norm, a.norm_dtype, static_cast<size_t>(h) * D + tid) : 0.f;
  // The token's rows are asked for before the state: loads come back in their order, and the decays are made from the rows while
  // the state is on its way (9.8 us against 10.2 the other way round).
  Four q, k;
  float gate, value;
  uint4 low[kTokenChunks];
  auto ask = [&](int t) __attribute__((always_inline)) {
    const bf16* from = a.proj + static_cast<size_t>(t) * a.proj_stride;
    const int d = tid < D ? tid : D - 1;
#pragma unroll
    for (int c = 0; c < kTokenChunks; ++c) {
      const int at = c * 32 + kq * 8;   // (a piece behind the rank, a multiple of 8, stands for the last one: its weights are zeros)
      low[c] = *reinterpret_cast<const uint4*>(from + a.low_at + (at < a.rank ? at : a.rank - 8));
    }
    value = to_float(from[a.v_at + h * D + d]);
    q = load_four(from + a.q_at + h * D + row);
    k = load_four(from + a.k_at + h * D + row);
    gate = to_float(from[a.g_at + h * D + d]);
  };
  ask(first);
  float4 s[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) s[i] = *reinterpret_cast<const float4*>(S + static_cast<size_t>(col0 + i * PER) * D);
  for (int t = first; t < first + count; ++t) {
    if (t > first) ask(t);
    if (tid < D) vs[tid] = value;
    if (decays) {
      floatx4 acc = {base[0], base[1], base[2], base[3]};
#pragma unroll
      for (int c = 0; c < kTokenChunks; ++c) {
        if (c >= chunks) break;   // (uniform)
        float xs[8];
        const uint32_t u[4] = {low[c].x, low[c].y, low[c].z, low[c].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          xs[2 * i] = __uint_as_float(u[i] << 16);
          xs[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
        }
        bf16x8 hi, mid, lo;
        tanh_in_three(xs, hi, mid, lo);
        acc = product_in_three(wv[c], hi, mid, lo, acc);
      }
      if (r16 == 0) {   // (all 16 columns of the operand are the token)
#pragma unroll
        for (int i = 0; i < 4; ++i) decay_s[wave * 16 + kq * 4 + i] = __expf(-__expf(acc[i]));
      }
    }
    __syncthreads();
    const float4 d4 = *reinterpret_cast<const float4*>(&decay_s[row]);
    const float dc[4] = {d4.x, d4.y, d4.z, d4.w};
    float o[LOADS < 4 ? 4 : LOADS] = {};
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const float v = vs[col0 + i * PER];
      float* si = reinterpret_cast<float*>(&s[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float kv = k.v[e] * v;
        o[i] = fmaf(fmaf(bonus[e], kv, si[e]), q.v[e], o[i]);
        si[e] = fmaf(si[e], dc[e], kv);
      }
    }
    if (t + 1 == first + count) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) *reinterpret_cast<float4*>(S + static_cast<size_t>(col0 + i * PER) * D) = s[i];
    }
#pragma unroll
    for (int i = 0; i < LOADS; i += 4) {
      float four[4] = {o[i], o[i + 1], o[i + 2], o[i + 3]};
      lanes_sum4<LPC>(four);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j < LOADS && lane % LPC == 0) os[col0 + (i + j) * PER] = four[j];
    }
    __syncthreads();
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < D / kWave; ++i) ss = fmaf(os[lane + i * kWave], os[lane + i * kWave], ss);
    ss = wave_sum(ss);
    const float scale = 1.f / sqrtf(ss / static_cast<float>(D) + a.eps);
    if (tid < D)
      a.out[static_cast<size_t>(t) * a.H * D + static_cast<size_t>(h) * D + tid] =
          float_to_bf16(os[tid] * scale * weight * (gate * (1.f / (1.f + expf(-gate)))));
    if (t + 1 < first + count) __syncthreads();   // the token's values, decays and sums have been read
  }
}

}  // namespace sa

using namespace sa;

extern "C" int sa_wkv_token_takes(int D, int rank, int64_t proj_stride, int q_at, int k_at, int low_at, int64_t state_stride,
                                  const void* proj, const void* state) {
  return (D == 64 || D == 128) && rank >= 8 && rank % 8 == 0 && rank <= 32 * kTokenChunks && proj_stride % 8 == 0 && q_at % 4 == 0 &&
         k_at % 4 == 0 && low_at % 8 == 0 && state_stride % 4 == 0 &&
         ((reinterpret_cast<uintptr_t>(proj) | reinterpret_cast<uintptr_t>(state)) & 15u) == 0;
}

extern "C" int sa_wkv_token(const void* proj, int64_t proj_stride, int q_at, int k_at, int v_at, int g_at, int low_at, int rank,
                            const void* decay_w, const void* base, int base_dtype, const void* bonus, int bonus_dtype,
                            const void* norm, int norm_dtype, float eps, int H, int D, float* state, int64_t state_stride,
                            const int* seq_meta, int num_seqs, void* out, hipStream_t stream) {
  if (num_seqs == 0) return 0;
  SA_REQUIRE(num_seqs > 0 && H > 0 && H <= 65535 && sa_wkv_token_takes(D, rank, proj_stride, q_at, k_at, low_at, state_stride, proj, state),
             "wkv_token: %d requests, %d heads of %d, rank %d are not taken", num_seqs, H, D, rank);
  SA_REQUIRE(proj != nullptr && decay_w != nullptr && base != nullptr && bonus != nullptr && norm != nullptr && state != nullptr &&
                 seq_meta != nullptr && out != nullptr,
             "wkv_token: a null pointer");
  const int64_t C = static_cast<int64_t>(H) * D;
  SA_REQUIRE(q_at >= 0 && k_at >= 0 && v_at >= 0 && g_at >= 0 && low_at >= 0 && proj_stride >= q_at + C && proj_stride >= k_at + C &&
                 proj_stride >= v_at + C && proj_stride >= g_at + C && proj_stride >= low_at + rank && state_stride >= C * D,
             "wkv_token: the projection rows or the state rows are too short");
  SA_REQUIRE((base_dtype == kF32 || base_dtype == kBF16) && (bonus_dtype == kF32 || bonus_dtype == kBF16) &&
                 (norm_dtype == kF32 || norm_dtype == kBF16) && eps >= 0.f,
             "wkv_token: unknown dtype");
  const WkvToken a{static_cast<const bf16*>(proj), proj_stride, q_at, k_at, v_at, g_at, low_at, rank,
                   static_cast<const bf16*>(decay_w), base, bonus, norm, base_dtype, bonus_dtype, norm_dtype, eps, H, state,
                   state_stride, seq_meta, static_cast<bf16*>(out)};
  if (D == 128) wkv_token_kernel<128><<<dim3(num_seqs, H), kTokenWaves * kWave, 0, stream>>>(a);
  else wkv_token_kernel<64><<<dim3(num_seqs, H), kTokenWaves * kWave, 0, stream>>>(a);
  return check_launch("wkv_token");
}
