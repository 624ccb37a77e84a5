// What latent attention makes of its projections before it scores anything, in one kernel:
//
//   queries   the last `rot_dims` entries of every head's vector turned by the token's position, in place
//   keys      the token's latent to unit RMS times a weight, the shared part turned, written as the row of a key page, and the
//             latent once more, transposed, into a value page
//
// Pairs (2p, 2p + 1) turn by position * freq[p]; angles, norm and products are 32-bit.  A workgroup of 16 waves takes 16 tokens;
// for the queries a thread keeps the angles of one piece of 8 entries for all the heads that it takes (a sine and cosine a token
// and pair, where a wave per token and head computed them once a head), for the keys a wave takes a token, a lane 8 entries of
// 16 bytes, and the values go through LDS so that 16 tokens that fill a page's 16 slots are written in pieces of 32 bytes.
// 2,047 tokens of 16 heads, latents of 512 and 64 turned: 11.5 us, by the wave-per-vector kernel in two launches 41 + 19.5; 8
// tokens 8.5, 5.3 + 13.4.  Bound by memory (13 MB) at 2,047 tokens, by its chain of waits at 8.
#include "api.h"
#include "common.h"
#include "eights.h"

namespace sa {

constexpr int kRowsTokens = 16;
struct LatentRows {
  bf16* q;
  const bf16* rows;
  int64_t q_stride, row_stride;
  const int* positions;
  const float* freq;
  const void* weight;
  const int64_t* slots;
  bf16 *k_pages, *v_pages;
  int T, H, R, dr, rot_dims, page_size, w_dtype;
  float mult, eps;
};

// Heads that a workgroup's threads turn at a time, and how many times one after the other; further heads are other workgroups'.
// (One token, 64 entries turned, us, this kernel / the wave-per-vector kernel in two launches: 16 heads 4.5 / 11.2, 64 7.6 / 11.2,
// 128 8.2 / 11.3, 512 9.0 / 11.5; one workgroup for all heads took 11.8 at 128 and 38 at 512.)
constexpr int kHeadsInTurn = 8;
__host__ __device__ constexpr int query_groups(int rot_dims) { return 1024 / (rot_dims / 8 * kRowsTokens); }

struct Turn {
  float c[4], s[4];
};
__device__ __forceinline__ Turn turn_of(float pos, const float* freq, float mult) {
  Turn t;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    sincosf(pos * freq[i], &t.s[i], &t.c[i]);
    t.s[i] *= mult;
    t.c[i] *= mult;
  }
  return t;
}
__device__ __forceinline__ Eight turned(const Eight& x, const Turn& t) {
  Eight y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    y.v[2 * i] = x.v[2 * i] * t.c[i] - x.v[2 * i + 1] * t.s[i];
    y.v[2 * i + 1] = x.v[2 * i + 1] * t.c[i] + x.v[2 * i] * t.s[i];
  }
  return y;
}

// NP: pieces of 512 entries of the latent.
template <int NP>
__global__ __launch_bounds__(1024) void latent_rows_kernel(LatentRows a) {
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, t0 = blockIdx.x * kRowsTokens;
  const int unit = a.R + a.dr;
  if (blockIdx.y > 0) {
    const int pieces = a.rot_dims / 8, groups = query_groups(a.rot_dims), first = (blockIdx.y - 1) * groups * kHeadsInTurn;
    const int end = first + groups * kHeadsInTurn < a.H ? first + groups * kHeadsInTurn : a.H;
    const int piece = tid % pieces, t = t0 + (tid / pieces) % kRowsTokens, group = tid / (pieces * kRowsTokens);
    if (t >= a.T || group >= groups) return;
    const Turn turn = turn_of(static_cast<float>(a.positions[t]), a.freq + piece * 4, a.mult);
    bf16* at = a.q + static_cast<size_t>(t) * a.q_stride + a.R + piece * 8;
#pragma unroll 2
    for (int h = first + group; h < end; h += groups) {
      bf16* p = at + static_cast<size_t>(h) * unit;
      store_eight(p, turned(load_eight(p), turn));
    }
    return;
  }
  extern __shared__ __align__(16) bf16 values[];   // [16 tokens][R]
  __shared__ int64_t slot_s[kRowsTokens];
  const int t = t0 + wave;
  const int64_t slot = t < a.T ? a.slots[t] : -1;
  if (lane == 0) slot_s[wave] = slot;
  if (slot >= 0) {
    const bf16* row = a.rows + static_cast<size_t>(t) * a.row_stride;
    Eight x[NP], w[NP];
    const int shared_at = lane * 8 < a.dr ? lane * 8 : 0;
    const Eight part = load_eight(row + a.R + shared_at);
    const float pos = static_cast<float>(a.positions[t]);
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {   // (a piece behind the latent stands for the last one)
      const int d = (p * kWave + lane) * 8, at = d < a.R ? d : a.R - 8;
      x[p] = load_eight(row + at);
      w[p] = a.w_dtype == kF32 ? load_eight(static_cast<const float*>(a.weight) + at) : load_eight(static_cast<const bf16*>(a.weight) + at);
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      float q = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) q = fmaf(x[p].v[e], x[p].v[e], q);
      ss += (p * kWave + lane) * 8 < a.R ? q : 0.f;
    }
    ss = wave_sum(ss);
    const float r = 1.f / sqrtf(ss / static_cast<float>(a.R) + a.eps);
    const int koff = static_cast<int>(slot % a.page_size);
    bf16* page = a.k_pages + (slot / a.page_size) * a.page_size * unit;
    const bool tiled = keys_tiled(a.page_size, unit);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int d = (p * kWave + lane) * 8;
      if (d >= a.R) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[p].v[e] = x[p].v[e] * r * w[p].v[e];
      store_eight(page + key_index(tiled, a.page_size, unit, koff, d), x[p]);
      store_eight(values + static_cast<size_t>(wave) * a.R + d, x[p]);
    }
    if (lane * 8 < a.dr)
      store_eight(page + key_index(tiled, a.page_size, unit, koff, a.R + lane * 8),
                  lane * 8 < a.rot_dims ? turned(part, turn_of(pos, a.freq + lane * 4, a.mult)) : part);
  }
  __syncthreads();
  const int64_t s0 = slot_s[0];
  bool page_full = s0 >= 0 && s0 % a.page_size % 16 == 0;   // 16 neighbouring slots of one page
#pragma unroll
  for (int i = 1; i < kRowsTokens; ++i) page_full = page_full && slot_s[i] == s0 + i;
  if (page_full && a.page_size % 16 == 0) {
    bf16* to = a.v_pages + (s0 / a.page_size) * a.page_size * a.R + s0 % a.page_size;
    for (int d = tid; d < a.R; d += 1024) {
      uint32_t u[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        u[i] = static_cast<uint32_t>(values[2 * i * a.R + d].bits) | (static_cast<uint32_t>(values[(2 * i + 1) * a.R + d].bits) << 16);
      uint4* p = reinterpret_cast<uint4*>(to + static_cast<size_t>(d) * a.page_size);
      p[0] = uint4{u[0], u[1], u[2], u[3]};
      p[1] = uint4{u[4], u[5], u[6], u[7]};
    }
    return;
  }
  if (slot < 0) return;
  bf16* to = a.v_pages + (slot / a.page_size) * a.page_size * a.R + slot % a.page_size;
  for (int d = lane; d < a.R; d += kWave) to[static_cast<size_t>(d) * a.page_size] = values[wave * a.R + d];
}

}  // namespace sa

using namespace sa;

extern "C" int sa_latent_rows_takes(int H, int R, int dr, int rot_dims, int page_size, int64_t q_stride, int64_t row_stride,
                                    const void* q, const void* rows, const void* weight, const void* k_pages, const void* v_pages) {
  const int pieces = rot_dims / 8;
  return H >= 1 && H <= 65535 && R >= 8 && R % 8 == 0 && R <= 1024 && dr >= 8 && dr % 8 == 0 && dr <= 8 * kWave && rot_dims >= 8 && rot_dims % 8 == 0 &&
         rot_dims <= dr && pieces * kRowsTokens <= 1024 && page_size >= 1 && q_stride % 8 == 0 && row_stride % 8 == 0 &&
         ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(rows) | reinterpret_cast<uintptr_t>(weight) |
           reinterpret_cast<uintptr_t>(k_pages) | reinterpret_cast<uintptr_t>(v_pages)) & 15u) == 0;
}

extern "C" int sa_latent_rows(void* q, int64_t q_stride, const void* rows, int64_t row_stride, const int* positions, const float* freq,
                              int rot_dims, float mult, const void* weight, int w_dtype, float eps, const int64_t* slots, void* k_pages,
                              void* v_pages, int T, int H, int R, int dr, int page_size, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && sa_latent_rows_takes(H, R, dr, rot_dims, page_size, q_stride, row_stride, q, rows, weight, k_pages, v_pages),
             "latent_rows: %d heads, latents of %d, %d shared entries of which %d turn are not taken", H, R, dr, rot_dims);
  SA_REQUIRE(q != nullptr && rows != nullptr && positions != nullptr && freq != nullptr && weight != nullptr && slots != nullptr &&
                 k_pages != nullptr && v_pages != nullptr,
             "latent_rows: a null pointer");
  SA_REQUIRE(q_stride >= static_cast<int64_t>(H) * (R + dr) && row_stride >= R + dr && eps >= 0.f && (w_dtype == kF32 || w_dtype == kBF16),
             "latent_rows: rows too short, or an unknown dtype");
  const LatentRows a{static_cast<bf16*>(q), static_cast<const bf16*>(rows), q_stride, row_stride, positions, freq, weight, slots,
                     static_cast<bf16*>(k_pages), static_cast<bf16*>(v_pages), T, H, R, dr, rot_dims, page_size, w_dtype, mult, eps};
  const int heads = query_groups(rot_dims) * kHeadsInTurn;
  const dim3 grid((T + kRowsTokens - 1) / kRowsTokens, 1 + (H + heads - 1) / heads);
  const size_t lds = static_cast<size_t>(kRowsTokens) * R * sizeof(bf16);
  if (R <= 512) latent_rows_kernel<1><<<grid, 1024, lds, stream>>>(a);
  else latent_rows_kernel<2><<<grid, 1024, lds, stream>>>(a);
  return check_launch("latent_rows");
}
