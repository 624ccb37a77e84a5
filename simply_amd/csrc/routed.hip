// A feed-forward of routed experts over a ragged batch of tokens.
//
//   route_few_kernel      for a handful of tokens: the router's product, its choice and the sort in one launch
//   route_kernel          softmax of the router's logits, the `top` largest scores and their experts
//   sort_kernel           the (token, choice) pairs in the order of their experts, cut into tiles of rows of one expert
//   expert_product_kernel h = act(Wg[e] x) * (Wu[e] x) for every pair, rows in the sorted order; then
//                         y = Wd[e] h, one row per pair (in the pairs' own order)
//   combine_kernel        out[t] = sum_k weight[t, k] y[t, k] + sigmoid(s[t]) * shared[t]
//
// Nothing comes back to the host between them: the tiles are found on the device, and the grid of the expert
// kernels is sized for the most tiles that the pairs can make.  Every pair's row is computed by itself, with sums
// in an order that depends on the sizes alone, so a token's result does not depend on the batch.  Scores are
// 32-bit; the products are bfloat16 on the matrix cores (32-bit accumulation) or 32-bit on the vector unit.
#include <climits>

#include "api.h"
#include "common.h"

namespace sa {

constexpr int kRouteSlots = 8;    // experts per lane: up to 512 experts
constexpr int kTileRowsMax = 64;  // rows of a tile: 16 (one MFMA operand) or 64 (four, which share the weights' operands),
constexpr int kTileRowsWide = 128;   // or 128, for the wide product kernel alone
constexpr int kGridMax = 65535;      // a grid's second and third index

// A wave per token.  scores = softmax(logits); `top` times the largest score that is left (of equal ones the lowest
// index); weight = score * scale.  SLOTS: experts a lane holds.
template <int SLOTS>
__device__ __forceinline__ void choose_plain(const float* __restrict__ logits, int E, int top, float scale, int* experts,
                                             float* weights) {
  const int lane = threadIdx.x % kWave;
  float z[SLOTS];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    const int e = lane + i * kWave;
    z[i] = e < E ? logits[e] : -INFINITY;
    mx = fmaxf(mx, z[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    z[i] = (lane + i * kWave) < E ? expf(z[i] - mx) : -1.f;   // (a score is never negative: -1 marks what is taken or absent)
    sum += z[i] > 0.f ? z[i] : 0.f;
  }
  sum = wave_sum(sum);
  for (int r = 0; r < top; ++r) {
    float best = -1.f;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) best = fmaxf(best, z[i]);
    best = wave_max(best);
    float mine = 1e9f;
#pragma unroll
    for (int i = SLOTS - 1; i >= 0; --i)
      if (z[i] == best) mine = static_cast<float>(lane + i * kWave);
    const float first = -wave_max(-mine);
    const int e = first < static_cast<float>(E) ? static_cast<int>(first) : E - 1;   // (logits that are no numbers: some expert)
#pragma unroll
    for (int i = 0; i < SLOTS; ++i)
      if (lane + i * kWave == e) z[i] = -1.f;
    if (lane == 0) {
      experts[r] = e;
      weights[r] = best / sum * scale;
    }
  }
}

__global__ __launch_bounds__(kWave) void route_kernel(const float* __restrict__ logits, int64_t stride, int E, int top,
                                                      float scale, int* __restrict__ experts,
                                                      float* __restrict__ weights) {
  const size_t t = blockIdx.x;
  choose_plain<kRouteSlots>(logits + t * stride, E, top, scale, experts + t * top, weights + t * top);
}

// A wave per token, for routers with options.  bias[e] (or null) is added to the logits first.  Scores are sigmoids of the
// logits, (softmax 1) their softmax over all experts, or (softmax 2) the logits themselves, and the weights are then the
// chosen ones' softmax among themselves (times scale; no renorm).  The choice is made by score + correction[e] (correction null: by the score); the experts form `groups`
// equal groups of neighbours, a group's score is the sum of its two largest choice scores (group_best 2; of its only
// one, in groups of one) or the largest one (group_best 1), and only experts of the `keep` groups with the largest
// scores can be chosen (of equal ones the lowest index, for groups and for experts).  weight = score * scale without
// the correction, with renorm >= 0 divided by the chosen scores' sum + renorm.  Choice scores can be negative: what is
// taken or shut out is -inf.
struct RouterOptions {
  const void *bias, *correction;
  int bias_dtype, corr_dtype, groups, keep, softmax, group_best;
  float renorm;
};
// What a wave wrote to LDS that is its own, its other lanes read from here on (a wave's LDS accesses run in their order: this
// keeps the compiler to it, and no other wave is waited for).
__device__ __forceinline__ void wave_ordered() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// choice_s, group_s: SLOTS * 64 words of LDS of the wave's own.
template <int SLOTS>
__device__ __forceinline__ void choose_with_options(const float* __restrict__ logits, int E, int top, float scale,
                                                    const RouterOptions& o, float* choice_s, float* group_s, int* experts,
                                                    float* weights) {
  const int lane = threadIdx.x % kWave;
  float s[SLOTS], c[SLOTS];
  float mx = -INFINITY, sum = 0.f;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    const int e = lane + i * kWave;
    s[i] = e < E ? logits[e] : -INFINITY;
    if (o.bias != nullptr && e < E) s[i] += load_f(o.bias, o.bias_dtype, e);
    mx = fmaxf(mx, s[i]);
  }
  if (o.softmax == 1) {
    mx = wave_max(mx);
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      s[i] = lane + i * kWave < E ? expf(s[i] - mx) : 0.f;
      sum += s[i];
    }
    sum = wave_sum(sum);
  }
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    const int e = lane + i * kWave;
    c[i] = -INFINITY;
    if (e < E) {
      if (o.softmax != 2) s[i] = o.softmax ? s[i] / sum : 1.f / (1.f + expf(-s[i]));
      c[i] = o.correction != nullptr ? s[i] + load_f(o.correction, o.corr_dtype, e) : s[i];
      choice_s[e] = c[i];
    } else {
      s[i] = 0.f;
    }
  }
  if (o.groups > 1) {
    wave_ordered();
    const int per = E / o.groups;
    for (int g = lane; g < o.groups; g += kWave) {
      float a = -INFINITY, b = -INFINITY;   // the two largest of the group
      for (int k = 0; k < per; ++k) {
        const float v = choice_s[g * per + k];
        if (v > a) {
          b = a;
          a = v;
        } else if (v > b) {
          b = v;
        }
      }
      group_s[g] = per > 1 && o.group_best > 1 ? a + b : a;
    }
    wave_ordered();
    // the `keep` best groups, one after the other; lane 0 marks them by sign in LDS
    for (int r = 0; r < o.keep; ++r) {
      float best = -INFINITY;
      for (int g = lane; g < o.groups; g += kWave) best = fmaxf(best, group_s[g]);
      best = wave_max(best);
      float mine = static_cast<float>(o.groups - 1);
      for (int g = lane; g < o.groups; g += kWave)
        if (group_s[g] == best && static_cast<float>(g) < mine) mine = static_cast<float>(g);
      const int g_best = static_cast<int>(-wave_max(-mine));
      wave_ordered();
      if (lane == 0) group_s[g_best] = -INFINITY;   // taken: -inf marks a group that stays
      wave_ordered();
    }
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const int e = lane + i * kWave;
      if (e < E && group_s[e / per] != -INFINITY) c[i] = -INFINITY;
    }
  }
  wave_ordered();   // the choice scores in LDS have been read: the chosen scores take their place
  float total = 0.f;
  for (int r = 0; r < top; ++r) {
    float best = -INFINITY;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) best = fmaxf(best, c[i]);
    best = wave_max(best);
    float mine = 1e9f;
#pragma unroll
    for (int i = SLOTS - 1; i >= 0; --i)
      if (c[i] == best && lane + i * kWave < E) mine = static_cast<float>(lane + i * kWave);
    const float first = -wave_max(-mine);
    const int e = first < static_cast<float>(E) ? static_cast<int>(first) : E - 1;   // (logits that are no numbers: some expert)
    float w = 0.f;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i)
      if (lane + i * kWave == e) {
        c[i] = -INFINITY;
        w = s[i];
      }
    w = wave_sum(w);   // (one lane holds it, the others 0)
    total += w;
    if (lane == 0) {
      experts[r] = e;
      choice_s[r] = w;
    }
  }
  wave_ordered();
  if (o.softmax == 2) {
    float best = -INFINITY, among = 0.f;
    for (int r = 0; r < top; ++r) best = fmaxf(best, choice_s[r]);
    for (int r = 0; r < top; ++r) among += expf(choice_s[r] - best);
    for (int r = lane; r < top; r += kWave) weights[r] = expf(choice_s[r] - best) / among * scale;
    return;
  }
  const float by = o.renorm >= 0.f ? total + o.renorm : 1.f;
  for (int r = lane; r < top; r += kWave) weights[r] = choice_s[r] / by * scale;
}

__global__ __launch_bounds__(kWave) void route_choice_kernel(const float* __restrict__ logits, int64_t stride, int E,
                                                             int top, float scale, RouterOptions options,
                                                             int* __restrict__ experts, float* __restrict__ weights) {
  __shared__ float choice_s[kRouteSlots * kWave];
  __shared__ float group_s[kRouteSlots * kWave];
  const size_t t = blockIdx.x;
  choose_with_options<kRouteSlots>(logits + t * stride, E, top, scale, options, choice_s, group_s, experts + t * top,
                                   weights + t * top);
}

// One workgroup.  plan: [0] number of tiles; [1 .. 1 + 3 * max_tiles): per tile its expert, its first row in the sorted order
// and the number of its rows.  sorted [P]: pair indices by expert.
__global__ __launch_bounds__(1024) void sort_kernel(const int* __restrict__ experts, int P, int E,
                                                    int* __restrict__ sorted, int* __restrict__ plan, int max_tiles,
                                                    int kTileRows) {
  extern __shared__ int lds[];   // counts [E], offsets [E + 1], tile offsets [E + 1], cursors [E]
  int* counts = lds;
  int* offsets = lds + E;
  int* tiles = offsets + E + 1;
  int* cursor = tiles + E + 1;
  for (int e = threadIdx.x; e < E; e += blockDim.x) counts[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) atomicAdd(&counts[experts[p]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0, nt = 0;
    for (int e = 0; e < E; ++e) {
      offsets[e] = at;
      tiles[e] = nt;
      at += counts[e];
      nt += (counts[e] + kTileRows - 1) / kTileRows;
    }
    offsets[E] = at;
    tiles[E] = nt;
    plan[0] = nt < max_tiles ? nt : max_tiles;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    cursor[e] = 0;
    for (int i = 0; tiles[e] + i < tiles[e + 1]; ++i) {
      const int n = tiles[e] + i;
      if (n >= max_tiles) break;
      const int rows = counts[e] - i * kTileRows < kTileRows ? counts[e] - i * kTileRows : kTileRows;
      plan[1 + 3 * n] = e;
      plan[2 + 3 * n] = offsets[e] + i * kTileRows;
      plan[3 + 3 * n] = rows;
    }
  }
  __syncthreads();
  // (the order of an expert's rows among themselves is whatever the atomics give: every row is computed by itself)
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    const int e = experts[p];
    sorted[offsets[e] + atomicAdd(&cursor[e], 1)] = p;
  }
}

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

__device__ __forceinline__ bf16x8 load8(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

// The router of a step of at most 16 tokens and 128 experts, from the rows to the plan: logits = x . router^T, every token's
// choice, and the pairs in the order of their experts, in one workgroup of 16 waves.  Three launches that each have next to
// nothing to do become one: the product by itself took 4.5 us, the choice 7.0 and the sort 3.6 (8 tokens, 2,048 wide, 16
// experts), this kernel 9.6.  Bound by its chain of waits: rows and weights from L2, a sum over the waves through LDS, a
// token's choices one after the other, in code that the CU has to fetch (for up to 64 experts and pairs: a variant of half the size,
// SLOTS 1).  Meanwhile the other workgroups of the launch (DENSE) make the hidden rows of a shared feed-forward, which need no
// router: a workgroup per 16 columns, whose waves share K as in the product here.  Beside the experts' first product they cost 2.8 us
// (2,048 x 2,048), here nothing.
//   product   a wave takes 1 / 16 of K for every tile of 16 experts; the waves' sums are added up by halves
//   choice    wave t is token t's
//   sort      lane e counts expert e's pairs; an expert's pairs stay in their order
// logits [T, stride] (32-bit): the first E are the experts', what follows (a shared expert's score) is only written.
constexpr int kFewTokens = 16, kFewSlots = 2, kFewPairs = 128;
struct DenseHidden {
  const bf16* w;   // tiled; gated: the two factors' tiles in turn
  bf16* out;       // [T, N]
  int N, gated, act;
  float limit;
};
template <int SLOTS>
struct RouterScratch {
  float logits[kFewTokens][SLOTS * kWave + 16];
  float sums[kFewTokens][16 * 17];   // the waves' tiles of 16 experts x 16 tokens
  float choice[kFewTokens][SLOTS * kWave], group[kFewTokens][SLOTS * kWave];
  int pairs[SLOTS * kWave];
};
// An entry of the waves' tiles, added up by halves.  (One after the other, and with one chain of products a wave instead of two, logits
// were 1.06 to 1.3 times as far from 64 bits as the product kernel's, which has fewer waves; now 0.74 to 0.99 times, in the same time.)
__device__ __forceinline__ float waves_sum(const float (&sums)[kFewTokens][16 * 17], int at) {
  float s[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) s[k] = sums[k][at];
#pragma unroll
  for (int n = 8; n > 0; n /= 2)
#pragma unroll
    for (int k = 0; k < n; ++k) s[k] += s[k + n];
  return s[0];
}
constexpr int kDenseLds = 2 * kFewTokens * 16 * 17 * sizeof(float);   // the waves' sums of two tiles
template <int SLOTS>
__global__ __launch_bounds__(1024) void route_few_kernel(const bf16* __restrict__ x, int64_t x_stride, const bf16* __restrict__ w,
                                                         int T, int D, int rows, int E, int top, float scale, int plain,
                                                         RouterOptions options, float* __restrict__ logits,
                                                         int* __restrict__ experts, float* __restrict__ weights,
                                                         int* __restrict__ sorted, int* __restrict__ plan, DenseHidden dense) {
  extern __shared__ __align__(16) char few_lds[];
  RouterScratch<SLOTS>& l = *reinterpret_cast<RouterScratch<SLOTS>*>(few_lds);
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r = lane % 16, kq = lane / 16, chunks = D / 32;
  const int c0 = chunks * wave / 16, c1 = chunks * (wave + 1) / 16;
  const bf16* row = x + static_cast<size_t>(r < T ? r : T - 1) * x_stride + kq * 8;
  if (blockIdx.x > 0) {   // a tile of the shared feed-forward's hidden columns
    float (*sums)[kFewTokens][16 * 17] = reinterpret_cast<float (*)[kFewTokens][16 * 17]>(few_lds);
    const int n0 = (blockIdx.x - 1) * 16;
    const bf16* g = dense.w + static_cast<size_t>((blockIdx.x - 1) * (dense.gated ? 2 : 1)) * chunks * 512 + lane * 8;
    const bf16* u = dense.gated ? g + static_cast<size_t>(chunks) * 512 : g;
    floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    constexpr int kAhead = 4;
    for (int c = c0; c < c1; c += kAhead) {
      bf16x8 gv[kAhead], uv[kAhead], xv[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const int at = c + i < c1 ? c + i : c1 - 1;
        gv[i] = load8(g + static_cast<size_t>(at) * 512);
        uv[i] = load8(u + static_cast<size_t>(at) * 512);
        xv[i] = load8(row + at * 32);
      }
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        if (c + i >= c1) break;   // (uniform)
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gv[i], xv[i], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uv[i], xv[i], acc[1], 0, 0, 0);
      }
    }
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int v = 0; v < 4; ++v) sums[f][wave][(4 * kq + v) * 17 + r] = acc[f][v];   // [column][token]
    __syncthreads();
    const int n = tid % 16, t = tid / 16;
    if (tid >= 256 || t >= T || n0 + n >= dense.N) return;
    const float first = to_float(float_to_bf16(waves_sum(sums[0], n * 17 + t)));
    const float second = to_float(float_to_bf16(waves_sum(sums[1], n * 17 + t)));
    const float h = dense.gated ? gated_product(dense.act, dense.limit, first, second) : gated_activation(dense.act, first);
    dense.out[static_cast<size_t>(t) * dense.N + n0 + n] = float_to_bf16(h);
    return;
  }
  for (int n0 = 0; n0 < rows; n0 += 16) {
    const bf16* tile = w + static_cast<size_t>(n0 / 16) * chunks * 512 + lane * 8;
    floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    constexpr int kAhead = 4;
    for (int c = c0; c < c1; c += kAhead) {
      bf16x8 wv[kAhead], xv[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {   // (a chunk behind the range is read again and not used)
        const int at = c + i < c1 ? c + i : c1 - 1;
        wv[i] = load8(tile + static_cast<size_t>(at) * 512);
        xv[i] = load8(row + at * 32);
      }
#pragma unroll
      for (int i = 0; i < kAhead; ++i)
        if (c + i < c1) acc[i % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[i], xv[i], acc[i % 2], 0, 0, 0);   // (uniform)
    }
    acc[0] += acc[1];
    if (n0 > 0) __syncthreads();   // the tile before has been added up
#pragma unroll
    for (int v = 0; v < 4; ++v) l.sums[wave][(4 * kq + v) * 17 + r] = acc[0][v];   // [expert][token]
    __syncthreads();
    if (tid < 256) {
      const int n = tid % 16, t = tid / 16;
      const float sum = waves_sum(l.sums, n * 17 + t);
      l.logits[t][n0 + n] = sum;
      if (t < T && n0 + n < rows) logits[static_cast<size_t>(t) * rows + n0 + n] = sum;
    }
  }
  __syncthreads();
  if (wave < T) {
    const int t = wave;
    int* chosen = l.pairs + t * top;
    float* weight = l.sums[wave];   // (the sums have been read)
    if (plain) choose_plain<SLOTS>(l.logits[t], E, top, scale, chosen, weight);
    else choose_with_options<SLOTS>(l.logits[t], E, top, scale, options, l.choice[wave], l.group[wave], chosen, weight);
    wave_ordered();
    for (int k = lane; k < top; k += kWave) {
      experts[t * top + k] = chosen[k];
      weights[t * top + k] = weight[k];
    }
  }
  __syncthreads();
  if (wave != 0) return;
  // A lane has pairs lane, lane + 64 and experts lane, lane + 64; every pair's expert passes by all lanes once (a lane read: no
  // chain of LDS reads, no prefix sums).
  const int P = T * top;
  int mine[SLOTS], place[SLOTS] = {}, count[SLOTS] = {}, below[SLOTS] = {};
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) mine[i] = lane + i * kWave < P ? l.pairs[lane + i * kWave] : -1;
#pragma unroll
  for (int j = 0; j < SLOTS; ++j)
    for (int q = 0; q < kWave && j * kWave + q < P; ++q) {
      const int e = __builtin_amdgcn_readlane(mine[j], q);
#pragma unroll
      for (int i = 0; i < SLOTS; ++i) {
        place[i] += e < mine[i] || (e == mine[i] && j * kWave + q < lane + i * kWave) ? 1 : 0;
        count[i] += e == lane + i * kWave ? 1 : 0;
        below[i] += e < lane + i * kWave ? 1 : 0;
      }
    }
  int before = 0;   // tiles of the experts before
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    const int tiles = (count[i] + 15) / 16, most = 1 + (SLOTS * kWave - 1) / 16;
    int n = before;
    for (int k = 1; k <= most; ++k) {   // (a second tile only where logits that are no numbers gave one expert to a token twice)
      const uint64_t has = __ballot(tiles >= k);
      if (has == 0) break;
      n += __popcll(has & ((uint64_t{1} << lane) - 1));
      before += __popcll(has);
    }
    for (int k = 0; k < tiles; ++k) {
      const int left = count[i] - k * 16;
      plan[1 + 3 * (n + k)] = lane + i * kWave;
      plan[2 + 3 * (n + k)] = below[i] + k * 16;
      plan[3 + 3 * (n + k)] = left < 16 ? left : 16;
    }
    if (lane + i * kWave < P) sorted[place[i]] = lane + i * kWave;
  }
  if (lane == 0) plan[0] = before;
}

// h[row, f] = act(x[token] . Wg[e, f]) * (x[token] . Wu[e, f]); GATED false: y[pair, n] = h[row] . Wd[e, n].
// A workgroup of one wave takes one tile of rows and 16 columns (for all RT sub-tiles of 16 rows): nothing is shared between
// waves, and small workgroups even out over the CUs, of which the few experts that a decode step reads would give some two or
// three workgroups of four waves and others none.
// bfloat16: the weights are tiled ([E][N / 16][K / 32][64][8], see the product kernels), a wave's operands are one
// 16-byte load a lane (rows that are not 16-byte aligned are read element by element); 32-bit: row-major weights
// [E][N][K], a lane per (row, column) of the tile in turn.
// SHARED (bfloat16, few tokens, products without a gate): the first tile of the grid is the shared feed-forward's, all tokens' rows
// against its own weights: a launch less a layer, and its 8 MB ride along with the experts' (8 tokens, feed-forwards of 2,048 x
// 2,048, 16 experts: 17.5 + 5.5 us before and 19.3 now).
struct SharedExpert {
  const bf16* a;
  const bf16* w;
  void* out;
  int64_t a_stride, out_stride;
  int N, K, rows;
};
template <typename T, bool GATED, int RT, bool SHARED = false>
__global__ __launch_bounds__(kWave) void expert_product_kernel(
    const T* __restrict__ a, int64_t a_stride, int a_by_token, int top, const T* __restrict__ w1, const T* __restrict__ w2,
    int N, int K, const int* __restrict__ sorted, const int* __restrict__ plan, int act, float limit,
    void* __restrict__ out, int64_t out_stride, int out_by_pair, int activate, SharedExpert sh) {
  // activate (without a second weight): out[row] = act(a . w1[e]^T) in a's type instead of the 32-bit product
  int tile = blockIdx.z * kGridMax + blockIdx.y;   // (gridDim would be one more load in front of everything)
  const bool shared = SHARED && tile == 0;
  if constexpr (SHARED) --tile;
  const int lane = threadIdx.x, n0 = blockIdx.x * 16;
  int e = 0, row0 = 0, rows;
  if (shared) {
    rows = sh.rows;
    if constexpr (SHARED) {
      a = sh.a, a_stride = sh.a_stride, out = sh.out, out_stride = sh.out_stride;
      N = sh.N, K = sh.K, out_by_pair = 0;
    }
  } else {
    if (tile >= plan[0]) return;
    e = plan[1 + 3 * tile], row0 = plan[2 + 3 * tile], rows = plan[3 + 3 * tile];
  }
  if constexpr (SHARED) if (n0 >= N) return;   // (the grid covers the wider of the two)
  if constexpr (sizeof(T) == 2) {
    const int Nt = (N + 15) / 16, Kt = (K + 31) / 32;
    const int r = lane % 16, kq = lane / 16;
    const bool aligned = a_stride % 8 == 0;
    const T* arow[RT];
    int pairs[RT];
#pragma unroll
    for (int s = 0; s < RT; ++s) {
      const int rr = s * 16 + r < rows ? s * 16 + r : rows - 1;
      pairs[s] = shared ? rr : sorted[row0 + rr];
      arow[s] = a + static_cast<size_t>(a_by_token && !shared ? pairs[s] / top : row0 + rr) * a_stride;
    }
    const size_t wbase = (static_cast<size_t>(e) * Nt + n0 / 16) * Kt;
    const bf16* g = reinterpret_cast<const bf16*>(w1) + wbase * 512 + lane * 8;
    const bf16* u = GATED ? reinterpret_cast<const bf16*>(w2) + wbase * 512 + lane * 8 : nullptr;
    if constexpr (SHARED) {
      if (shared) {
        static_assert(!GATED, "the shared rows of gated products are the router's launch's");
        g = sh.w + wbase * 512 + lane * 8;
      }
    }
    floatx4 accg[RT], accu[RT];
#pragma unroll
    for (int s = 0; s < RT; ++s) accg[s] = accu[s] = floatx4{0.f, 0.f, 0.f, 0.f};
    // Whole k tiles of aligned rows: two sets of four, so that one set's loads are under way while the other is multiplied.
    // Loads behind the last tile ask for it again; the products go in the order of k.  (Weights of 16 experts of 2,048 x 2,048
    // from HBM, top 2, gate and up + down: 8 tokens 43.3 + 26.8 us with one set and workgroups of four waves, 37.0 + 22.8 with
    // one set, 45.1 + 26.9 with two sets, 33.7 + 18.0 with two sets and one wave, 5.1 TB/s; 1 token 17.6 + 11.5 and 9.4 + 7.6;
    // 64 tokens 50.5 + 29.3 and 52.8 + 29.7.  Sets of eight: 34.1 + 18.4.)
    int kt = 0;
    if (aligned && RT == 1) {
      const bf16* src = reinterpret_cast<const bf16*>(arow[0]) + kq * 8;
      constexpr int kAhead = 4;
      const int whole = K / 32;
      bf16x8 gv[2][kAhead], uv[2][kAhead], av[2][kAhead];
      auto load = [&](int set, int from) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          const int at = from + i < whole ? from + i : whole - 1;
          gv[set][i] = load8(g + static_cast<size_t>(at) * 512);
          if constexpr (GATED) uv[set][i] = load8(u + static_cast<size_t>(at) * 512);
          av[set][i] = load8(src + at * 32);
        }
      };
      auto multiply = [&](int set, int i) __attribute__((always_inline)) {
        accg[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gv[set][i], av[set][i], accg[0], 0, 0, 0);
        if constexpr (GATED) accu[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uv[set][i], av[set][i], accu[0], 0, 0, 0);
      };
      if (whole > 0) {
        load(0, 0);
        load(1, kAhead);
        for (; kt + 2 * kAhead <= whole; kt += 2 * kAhead) {
#pragma unroll
          for (int set = 0; set < 2; ++set) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) multiply(set, i);
            load(set, kt + (2 + set) * kAhead);
          }
        }
#pragma unroll
        for (int i = 0; i < 2 * kAhead; ++i)
          if (kt + i < whole) multiply(i / kAhead, i % kAhead);   // (uniform)
        kt = whole;
      }
    }
    for (; kt < Kt; ++kt) {
      const int k = kt * 32 + kq * 8;
      const bf16x8 gv = load8(g + static_cast<size_t>(kt) * 512);
      bf16x8 uv = gv;
      if constexpr (GATED) uv = load8(u + static_cast<size_t>(kt) * 512);
#pragma unroll
      for (int s = 0; s < RT; ++s) {
        if (s * 16 >= rows) break;   // (uniform: the tile's rows are)
        const bf16* src = reinterpret_cast<const bf16*>(arow[s]);
        bf16x8 av;
        if (aligned && k + 8 <= K) {
          av = load8(src + k);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i)
            av[i] = k + i < K ? __builtin_bit_cast(__bf16, src[k + i]) : static_cast<__bf16>(0.f);
        }
        // the weights' rows are the product's columns: C^T = W . A^T, a lane holds four columns of the output of
        // one token
        accg[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gv, av, accg[s], 0, 0, 0);
        if constexpr (GATED) accu[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uv, av, accu[s], 0, 0, 0);
      }
    }
    // lane: token s * 16 + lane % 16, output columns n0 + kq * 4 + i
#pragma unroll
    for (int s = 0; s < RT; ++s) {
      if (s * 16 + r >= rows) continue;
      const size_t orow = static_cast<size_t>(out_by_pair ? pairs[s] : row0 + s * 16 + r) * out_stride;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = n0 + kq * 4 + i;
        if (n >= N) continue;
        if constexpr (GATED) {
          const float v = gated_product(act, limit, to_float(float_to_bf16(accg[s][i])), to_float(float_to_bf16(accu[s][i])));
          static_cast<bf16*>(out)[orow + n] = float_to_bf16(v);
        } else if (activate) {
          static_cast<bf16*>(out)[orow + n] = float_to_bf16(gated_activation(act, to_float(float_to_bf16(accg[s][i]))));
        } else {
          static_cast<float*>(out)[orow + n] = accg[s][i];
        }
      }
    }
  } else {
    // 32-bit: 16 columns x the rows of the tile over the wave's 64 lanes, four rows at a time
    const int c = lane % 16, n = n0 + c;
    for (int r = lane / 16; r < rows; r += 4) {
      const int pair = sorted[row0 + r];
      const T* arow = a + static_cast<size_t>(a_by_token ? pair / top : row0 + r) * a_stride;
      if (n >= N) continue;
      const T* g = w1 + (static_cast<size_t>(e) * N + n) * K;
      float sg = 0.f, su = 0.f;
      for (int k = 0; k < K; ++k) sg = fmaf(to_float(arow[k]), to_float(g[k]), sg);
      const size_t orow = static_cast<size_t>(out_by_pair ? pair : row0 + r) * out_stride;
      if constexpr (GATED) {
        const T* u = w2 + (static_cast<size_t>(e) * N + n) * K;
        for (int k = 0; k < K; ++k) su = fmaf(to_float(arow[k]), to_float(u[k]), su);
        static_cast<float*>(out)[orow + n] = gated_product_exact(act, limit, sg, su);
      } else {
        static_cast<float*>(out)[orow + n] = activate ? gated_activation_exact(act, sg) : sg;
      }
    }
  }
}

// The same products for tiles of 64 rows (steps that bring an expert many rows), bfloat16: a workgroup takes the tile's
// rows and 128 columns, a wave 32 of them (two column tiles) for all four sub-tiles of 16 rows.  The rows' operands of
// 64 columns of K at a time go through LDS in operand order (every wave needs all of them: read from memory once
// instead of four times), asked for a chunk ahead into registers; the weights' operands come straight from their
// tiles.  A row's sums are those of the kernel above, in its order.
constexpr int kChunkK = 64;
template <bool GATED>
__global__ __launch_bounds__(256) void expert_product_rows64_kernel(
    const bf16* __restrict__ a, int64_t a_stride, int a_by_token, int top, const bf16* __restrict__ w1,
    const bf16* __restrict__ w2, int N, int K, const int* __restrict__ sorted, const int* __restrict__ plan, int act, float limit,
    void* __restrict__ out, int64_t out_stride, int out_by_pair, int activate) {
  __shared__ bf16x8 rows_lds[4][kChunkK / 32][kWave];   // [sub-tile of 16 rows][k tile of the chunk][lane]
  __shared__ int pair_of[kTileRowsMax];
  const int tile = blockIdx.x;
  if (tile >= plan[0]) return;
  const int e = plan[1 + 3 * tile], row0 = plan[2 + 3 * tile], rows = plan[3 + 3 * tile];
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int r = lane % 16, kq = lane / 16;
  const int n0 = (blockIdx.y * 4 + wave) * 32;
  const bool mine = n0 < N;   // (a wave without columns still stages rows and meets the barriers)
  if (tid < kTileRowsMax) pair_of[tid] = sorted[row0 + (tid < rows ? tid : rows - 1)];
  __syncthreads();
  const bool aligned = a_stride % 8 == 0;
  // staging: this thread's two pieces of 8 elements of a chunk, and where they go
  const bf16* src[2];
  int koff[2];
  bf16x8* dst[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int combo = wave + 4 * i, sub = combo / 2, kt = combo % 2;
    const int row = sub * 16 + r, rr = row < rows ? row : rows - 1;
    src[i] = a + static_cast<size_t>(a_by_token ? pair_of[rr] / top : row0 + rr) * a_stride;
    koff[i] = kt * 32 + kq * 8;
    dst[i] = &rows_lds[sub][kt][lane];
  }
  bf16x8 staged[2];
  auto fetch = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = c * kChunkK + koff[i];
      if (aligned && k + 8 <= K) {
        staged[i] = load8(src[i] + k);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          staged[i][j] = k + j < K ? __builtin_bit_cast(__bf16, src[i][k + j]) : static_cast<__bf16>(0.f);
      }
    }
  };
  const int Nt = (N + 15) / 16, Kt = (K + 31) / 32;
  const int nsub = (rows + 15) / 16;
  floatx4 accg[4][2], accu[4][2];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int j = 0; j < 2; ++j) accg[s][j] = accu[s][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int chunks = (K + kChunkK - 1) / kChunkK;
  fetch(0);
  for (int c = 0; c < chunks; ++c) {
    __syncthreads();   // the chunk before has been read
    *dst[0] = staged[0];
    *dst[1] = staged[1];
    __syncthreads();
    if (c + 1 < chunks) fetch(c + 1);
    if (!mine) continue;
#pragma unroll
    for (int kt = 0; kt < kChunkK / 32; ++kt) {
      const int ktg = c * (kChunkK / 32) + kt;
      if (ktg >= Kt) break;
      bf16x8 gv[2], uv[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int nt = n0 / 16 + j < Nt ? n0 / 16 + j : Nt - 1;
        const size_t at = ((static_cast<size_t>(e) * Nt + nt) * Kt + ktg) * 512 + lane * 8;
        gv[j] = load8(w1 + at);
        if constexpr (GATED) uv[j] = load8(w2 + at);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s >= nsub) break;
        const bf16x8 av = rows_lds[s][kt][lane];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          accg[s][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gv[j], av, accg[s][j], 0, 0, 0);
          if constexpr (GATED) accu[s][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uv[j], av, accu[s][j], 0, 0, 0);
        }
      }
    }
  }
  if (!mine) return;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int row = s * 16 + r;
    if (row >= rows) continue;
    const size_t orow = static_cast<size_t>(out_by_pair ? pair_of[row] : row0 + row) * out_stride;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = n0 + j * 16 + kq * 4 + i;
        if (n >= N) continue;
        if constexpr (GATED) {
          const float v = gated_product(act, limit, to_float(float_to_bf16(accg[s][j][i])), to_float(float_to_bf16(accu[s][j][i])));
          static_cast<bf16*>(out)[orow + n] = float_to_bf16(v);
        } else if (activate) {
          static_cast<bf16*>(out)[orow + n] =
              float_to_bf16(gated_activation(act, to_float(float_to_bf16(accg[s][j][i]))));
        } else {
          static_cast<float*>(out)[orow + n] = accg[s][j][i];
        }
      }
  }
}

// out[t, d] = sum_k weights[t, k] * y[t * top + k, d] (in the order of k) + sigmoid(gate[t]) * shared[t, d].
__global__ void combine_kernel(const float* __restrict__ y, const float* __restrict__ weights, int top,
                               const void* __restrict__ shared, int shared_dtype, int64_t shared_stride,
                               const float* __restrict__ gate, int64_t gate_stride, void* __restrict__ out, int out_dtype,
                               int64_t out_stride, int D) {
  const int t = blockIdx.y, d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= D) return;
  float v = 0.f;
  for (int k = 0; k < top; ++k)
    v = fmaf(weights[static_cast<size_t>(t) * top + k], y[(static_cast<size_t>(t) * top + k) * D + d], v);
  if (shared != nullptr) {
    const float s = load_f(shared, shared_dtype, static_cast<size_t>(t) * shared_stride + d);
    v += gate != nullptr ? s / (1.f + expf(-gate[static_cast<size_t>(t) * gate_stride])) : s;
  }
  store_f(out, out_dtype, static_cast<size_t>(t) * out_stride + d, v);
}

// The same, four entries a thread: D and the strides multiples of four, rows aligned.  Bound by memory: 2,047 tokens of two
// experts' 2,048 entries (50 MB) take 10.2 us, an entry a thread took 18.6.
template <typename ST, typename OT>
__global__ __launch_bounds__(256) void combine_fours_kernel(const float* __restrict__ y, const float* __restrict__ weights,
                                                            int top, const ST* __restrict__ shared, int64_t shared_stride,
                                                            const float* __restrict__ gate, int64_t gate_stride,
                                                            OT* __restrict__ out, int64_t out_stride, int D) {
  const int t = blockIdx.y, d = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (d >= D) return;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if (shared != nullptr) {   // (asked for first: under way with the experts' rows)
    const ST* from = shared + static_cast<size_t>(t) * shared_stride + d;
    if constexpr (sizeof(ST) == 4) {
      const float4 q = *reinterpret_cast<const float4*>(from);
      s[0] = q.x, s[1] = q.y, s[2] = q.z, s[3] = q.w;
    } else {
      struct __align__(8) Four { bf16 v[4]; };
      const Four q = *reinterpret_cast<const Four*>(from);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = to_float(q.v[i]);
    }
  }
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < top; ++k) {
    const float wk = weights[static_cast<size_t>(t) * top + k];
    const float4 q = *reinterpret_cast<const float4*>(y + (static_cast<size_t>(t) * top + k) * D + d);
    v[0] = fmaf(wk, q.x, v[0]), v[1] = fmaf(wk, q.y, v[1]), v[2] = fmaf(wk, q.z, v[2]), v[3] = fmaf(wk, q.w, v[3]);
  }
  if (shared != nullptr) {
    const float f = gate != nullptr ? 1.f + expf(-gate[static_cast<size_t>(t) * gate_stride]) : 1.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += gate != nullptr ? s[i] / f : s[i];
  }
  OT* to = out + static_cast<size_t>(t) * out_stride + d;
  if constexpr (sizeof(OT) == 4) {
    *reinterpret_cast<float4*>(to) = float4{v[0], v[1], v[2], v[3]};
  } else {
    struct __align__(8) Four { bf16 v[4]; };
    Four q;
#pragma unroll
    for (int i = 0; i < 4; ++i) q.v[i] = float_to_bf16(v[i]);
    *reinterpret_cast<Four*>(to) = q;
  }
}

}  // namespace sa

using namespace sa;

extern "C" int sa_route(const float* logits, int64_t stride, int T, int E, int top, float scale, int* experts,
                        float* weights, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && E > 0 && E <= kRouteSlots * kWave && top > 0 && top <= E && stride >= E,
             "route: bad sizes T=%d E=%d top=%d (at most %d experts)", T, E, top, kRouteSlots * kWave);
  SA_REQUIRE(logits != nullptr && experts != nullptr && weights != nullptr, "route: a null pointer");
  route_kernel<<<T, kWave, 0, stream>>>(logits, stride, E, top, scale, experts, weights);
  return check_launch("route");
}

extern "C" int sa_route_choice(const float* logits, int64_t stride, int T, int E, int top, float scale,
                               const void* bias, int bias_dtype, const void* correction, int corr_dtype, int groups, int keep, int softmax,
                               int group_best, float renorm, int* experts, float* weights, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && E > 0 && E <= kRouteSlots * kWave && top > 0 && stride >= E,
             "route_choice: bad sizes T=%d E=%d top=%d (at most %d experts)", T, E, top, kRouteSlots * kWave);
  SA_REQUIRE(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups,
             "route_choice: %d experts in %d groups of which %d stay", E, groups, keep);
  SA_REQUIRE(group_best == 1 || group_best == 2, "route_choice: a group's score is its largest or its two largest");
  SA_REQUIRE(top <= keep * (E / groups), "route_choice: %d experts cannot be chosen from %d groups of %d", top, keep,
             E / groups);
  SA_REQUIRE(correction == nullptr || corr_dtype == kF32 || corr_dtype == kBF16, "route_choice: unknown dtype %d",
             corr_dtype);
  SA_REQUIRE(bias == nullptr || bias_dtype == kF32 || bias_dtype == kBF16, "route_choice: unknown dtype %d", bias_dtype);
  SA_REQUIRE(softmax >= 0 && softmax <= 2 && (softmax != 2 || renorm < 0.f),
             "route_choice: scores %d (0 sigmoid, 1 softmax, 2 the chosen logits' softmax, which sums to 1 by itself)", softmax);
  route_choice_kernel<<<T, kWave, 0, stream>>>(
      logits, stride, E, top, scale,
      RouterOptions{bias, correction, bias_dtype, corr_dtype, groups, keep, softmax, group_best, renorm}, experts, weights);
  return check_launch("route_choice");
}

extern "C" int sa_route_few_takes(const void* x, int64_t x_stride, int T, int D, int rows, int E, int top) {
  // (the weights all go through one CU: 256 KiB of them take as long as the launch of the product that they save)
  return T >= 1 && T <= kFewTokens && D >= 32 && D % 32 == 0 && x_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && E >= 1 &&
         E <= kFewSlots * kWave && rows >= E && rows <= E + 16 && static_cast<int64_t>(rows) * D <= 128 * 1024 && top >= 1 &&
         top <= E && T * top <= kFewPairs;
}

// One CU against a product on many and two launches more.  What it costs above them in us, fitted to 300 sizes (logits on 1 to 9 tiles
// of 16 experts, 1 to 16 tokens, 1 to 128 pairs): a wave adds up and chooses for each token, tiles come one after the other, pairs pass
// by the sorting wave, the weights come through one CU, and more than 64 experts or pairs take the larger variant.  Few / three launches
// in us: 16 experts, top 2, 2,048 wide, 1 token 5.9 / 9.7, 8 7.8 / 11.1, 16 10.2 / 12.0; 32, top 4, 1,024 wide, 8 tokens 11.5 / 12.5, 12
// 13.5 / 12.7, 16 15.8 / 12.9; 64, top 6, 1,024 wide, 4 14.3 / 15.4, 8 17.4 / 15.7, 16 27.6 / 16.2; 128, top 8, 960 wide, 1 19.3 / 21.2,
// 8 30.0 / 21.9, 16 42.8 / 22.2.  (The line lies a little below the fit: of the sizes it takes none is more than 2 % behind.)
extern "C" int sa_route_few_pays(int T, int D, int rows, int E, int top) {
  const int tiles = (rows + 15) / 16;
  return 0.08 * T * tiles + 0.07 * T * top + 0.12 * tiles * D / 1024 + (E > kWave || T * top > kWave ? 1.3 : 0.0) < 4.4;
}

extern "C" int sa_route_few(const void* x, int64_t x_stride, const void* w, int T, int D, int rows, int E, int top, float scale,
                            int plain, const void* bias, int bias_dtype, const void* correction, int corr_dtype, int groups, int keep,
                            int softmax, int group_best, float renorm, float* logits, int* experts, float* weights, int* sorted,
                            int* plan, int plan_words, const void* dense_w, int dense_N, int dense_gated, int dense_act, float dense_limit,
                            void* dense_out, hipStream_t stream) {
  SA_REQUIRE(sa_route_few_takes(x, x_stride, T, D, rows, E, top) && x_stride >= D, "route_few: T=%d D=%d experts=%d top=%d are not taken", T,
             D, E, top);
  SA_REQUIRE(x != nullptr && w != nullptr && logits != nullptr && experts != nullptr && weights != nullptr && sorted != nullptr &&
                 plan != nullptr && plan_words >= 1 + 3 * sa_expert_tiles_max(T * top, E, 16),
             "route_few: a null pointer, or a plan too short");
  SA_REQUIRE(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups && (group_best == 1 || group_best == 2) &&
                 top <= keep * (E / groups) && softmax >= 0 && softmax <= 2 && (softmax != 2 || renorm < 0.f),
             "route_few: %d experts in %d groups of which %d stay, scores %d", E, groups, keep, softmax);
  SA_REQUIRE((correction == nullptr || corr_dtype == kF32 || corr_dtype == kBF16) &&
                 (bias == nullptr || bias_dtype == kF32 || bias_dtype == kBF16),
             "route_few: unknown dtype");
  SA_REQUIRE(dense_w == nullptr || (dense_out != nullptr && dense_N > 0 && dense_act >= 0 &&
                                    dense_act < (dense_gated ? kNumGatedRules : kNumActivations) &&
                                    (dense_act != kActClampedGlu || dense_limit > 0.f)),
             "route_few: a shared feed-forward of %d columns, activation %d", dense_N, dense_act);
  const DenseHidden dense{static_cast<const bf16*>(dense_w), static_cast<bf16*>(dense_out), dense_N, dense_gated, dense_act, dense_limit};
  const int blocks = 1 + (dense_w != nullptr ? (dense_N + 15) / 16 : 0);
#define SA_ROUTE_FEW(SLOTS)                                                                                                          \
  route_few_kernel<SLOTS><<<blocks, 1024, sizeof(RouterScratch<SLOTS>) > kDenseLds ? sizeof(RouterScratch<SLOTS>) : kDenseLds, stream>>>( \
      static_cast<const bf16*>(x), x_stride, static_cast<const bf16*>(w), T, D, rows, E, top, scale, plain,                            \
      RouterOptions{bias, correction, bias_dtype, corr_dtype, groups, keep, softmax, group_best, renorm}, logits, experts, weights,    \
      sorted, plan, dense)
  if (E <= kWave && T * top <= kWave) SA_ROUTE_FEW(1);
  else SA_ROUTE_FEW(2);
#undef SA_ROUTE_FEW
  return check_launch("route_few");
}

extern "C" int sa_expert_tiles_max(int P, int E, int tile_rows) {
  return (P + tile_rows - 1) / tile_rows + (E < P ? E : P);
}

extern "C" int sa_expert_tile_rows(int P, int E, int D, int F, int dtype, int64_t a_stride, const void* a) {
  alignas(16) static const char aligned_stand_in[16] = {};   // (weights and results are whole tensors)
  const void* p = aligned_stand_in;
  const bool wide = dtype == kBF16 && gemm_wide_routed_takes(F, D, a_stride, P, F, a, p, p, p, kTileRowsWide) &&
                    gemm_wide_routed_takes(D, F, F, P, D, p, p, nullptr, p, kTileRowsWide);
  // Rows that an expert gets on average: from 12 on some need a second tile of 16, which reads the weights again (2,048 x
  // 2,048, 16 experts: 8 rows 63 us with tiles of 16 and 72 with the wide kernel's 64; 16 rows 105 and 72); the kernel of 64
  // rows here is ahead from 32 on.
  if (P < (wide ? 12 : 32) * static_cast<int64_t>(E)) return 16;
  // Tiles of 128 x 256, one a CU, instead of 64 x 128, two a CU, halve what a CU fetches; what they cost is rounds: half as many
  // columns of tiles, and a last round that may be nearly empty.  With 2,048 columns or more in both products they are ahead from
  // nearly 64 rows an expert on; with fewer in one of them that product does not fill the CUs until there are many tiles of rows, and
  // only an expert so large that its products are long makes up for it (figures: gemm_wide_routed).
  const double mib = 4.0 * D * F / (1 << 20);   // of gate and up
  const int from = D >= 2048 && F >= 2048 ? 60 : mib >= 32 ? 128 : mib >= 16 ? 320 : INT_MAX;
  return wide && P >= from * static_cast<int64_t>(E) && sa_expert_tiles_max(P, E, kTileRowsWide) <= kGridMax ? kTileRowsWide : kTileRowsMax;
}

extern "C" int sa_expert_sort(const int* experts, int P, int E, int tile_rows, int* sorted, int* plan, int plan_words,
                              hipStream_t stream) {
  if (P == 0) return 0;
  SA_REQUIRE(tile_rows == 16 || tile_rows == kTileRowsMax || tile_rows == kTileRowsWide, "expert_sort: tiles of 16, %d or %d rows",
             kTileRowsMax, kTileRowsWide);
  const int max_tiles = sa_expert_tiles_max(P, E, tile_rows);
  SA_REQUIRE(P > 0 && E > 0 && E <= 4096 && P < (1 << 26), "expert_sort: bad sizes P=%d E=%d", P, E);
  SA_REQUIRE(plan_words >= 1 + 3 * max_tiles, "expert_sort: the plan needs %d words", 1 + 3 * max_tiles);
  SA_REQUIRE(experts != nullptr && sorted != nullptr && plan != nullptr, "expert_sort: a null pointer");
  const int threads = P >= 1024 ? 1024 : ((P + kWave - 1) / kWave) * kWave;
  sort_kernel<<<1, threads, (4 * E + 2) * sizeof(int), stream>>>(experts, P, E, sorted, plan, max_tiles, tile_rows);
  return check_launch("expert_sort");
}

extern "C" int sa_expert_product(const void* a, int dtype, int64_t a_stride, int a_by_token, int top, const void* w1,
                                 const void* w2, int N, int K, const int* sorted, const int* plan, int P, int E,
                                 int tile_rows, int act, float limit, void* out, int64_t out_stride, int out_by_pair, int activate,
                                 hipStream_t stream) {
  if (P == 0) return 0;
  SA_REQUIRE(!activate || w2 == nullptr, "expert_product: a gated product has its activation already");
  SA_REQUIRE(P > 0 && E > 0 && N > 0 && K > 0 && top > 0 && a_stride >= K && out_stride >= N,
             "expert_product: bad sizes P=%d E=%d N=%d K=%d", P, E, N, K);
  SA_REQUIRE(a != nullptr && w1 != nullptr && sorted != nullptr && plan != nullptr && out != nullptr,
             "expert_product: a null pointer");
  SA_REQUIRE(act >= 0 && act < (w2 != nullptr ? kNumGatedRules : kNumActivations), "expert_product: unknown activation %d", act);
  SA_REQUIRE(act != kActClampedGlu || limit > 0.f, "expert_product: the clamped gated product needs a positive limit");
  SA_REQUIRE(dtype == kF32 || dtype == kBF16, "expert_product: unknown dtype %d", dtype);
  SA_REQUIRE(tile_rows == 16 || tile_rows == kTileRowsMax || tile_rows == kTileRowsWide,
             "expert_product: tiles of 16, %d or %d rows", kTileRowsMax, kTileRowsWide);
  const int tiles = sa_expert_tiles_max(P, E, tile_rows);
  // (the grid's second and third index go to 65,535; tiles of the kernels of 16 and 64 rows here are not limited by that)
  const int tiles_y = tiles < kGridMax ? tiles : kGridMax, tiles_z = (tiles + tiles_y - 1) / tiles_y;
  const bool gated = w2 != nullptr;
#define SA_EXPERT(T, G, RT)                                                                                            \
  expert_product_kernel<T, G, RT><<<dim3((N + 15) / 16, tiles_y, tiles_z), kWave, 0, stream>>>(                          \
      static_cast<const T*>(a), a_stride, a_by_token, top, static_cast<const T*>(w1), static_cast<const T*>(w2), N, K,   \
      sorted, plan, act, limit, out, out_stride, out_by_pair, activate, SharedExpert{})
  // Tiles of 64 and 128 rows go to the wide product kernel where it takes the operands; the others to the kernel of 64 rows here.
  const bool by_wide = dtype == kBF16 && tile_rows != 16 && tiles <= kGridMax && ((gated || activate) ? !out_by_pair : out_by_pair != 0) &&
                       gemm_wide_routed_takes(N, K, a_stride, a_by_token ? (P + top - 1) / top : P, out_stride, a, w1, w2, out, tile_rows);
  SA_REQUIRE(by_wide || tile_rows != kTileRowsWide, "expert_product: tiles of %d rows need aligned bfloat16 operands, K in multiples of 64",
             kTileRowsWide);
  if (by_wide)
    return gemm_wide_routed(a, a_stride, w1, w2, gated || activate ? out : nullptr,
                            gated || activate ? nullptr : static_cast<float*>(out), out_stride, tiles, N, K, tile_rows, plan, sorted,
                            a_by_token, top, gated ? act : activate ? act + 1 : 0, limit, stream);
  if (dtype == kBF16) {
    if (tile_rows == 16) {
      if (gated) SA_EXPERT(bf16, true, 1);
      else SA_EXPERT(bf16, false, 1);
    } else {
      const dim3 wide(tiles, (N + 127) / 128);
      if (gated)
        expert_product_rows64_kernel<true><<<wide, 256, 0, stream>>>(
            static_cast<const bf16*>(a), a_stride, a_by_token, top, static_cast<const bf16*>(w1),
            static_cast<const bf16*>(w2), N, K, sorted, plan, act, limit, out, out_stride, out_by_pair, 0);
      else
        expert_product_rows64_kernel<false><<<wide, 256, 0, stream>>>(
            static_cast<const bf16*>(a), a_stride, a_by_token, top, static_cast<const bf16*>(w1), nullptr, N, K, sorted,
            plan, act, limit, out, out_stride, out_by_pair, activate);
    }
  } else {
    if (gated) SA_EXPERT(float, true, 1);
    else SA_EXPERT(float, false, 1);
  }
#undef SA_EXPERT
  return check_launch("expert_product");
}

extern "C" int sa_expert_product_shared(const void* h, int64_t h_stride, int top, const void* w, int N, int K, const int* sorted,
                                        const int* plan, int P, int E, void* y, int64_t y_stride, const void* shared_h,
                                        int64_t shared_h_stride, const void* shared_w, int shared_N, int shared_K, int T, void* shared_y,
                                        int64_t shared_y_stride, hipStream_t stream) {
  SA_REQUIRE(P > 0 && E > 0 && N > 0 && K > 0 && top > 0 && h_stride >= K && y_stride >= N && T > 0 && T <= 16 && P == T * top &&
                 shared_N > 0 && shared_K > 0 && shared_h_stride >= shared_K && shared_y_stride >= shared_N,
             "expert_product_shared: bad sizes P=%d E=%d N=%d K=%d, %d tokens (at most 16), N=%d K=%d", P, E, N, K, T, shared_N, shared_K);
  SA_REQUIRE(h != nullptr && w != nullptr && sorted != nullptr && plan != nullptr && y != nullptr && shared_h != nullptr &&
                 shared_w != nullptr && shared_y != nullptr,
             "expert_product_shared: a null pointer");
  const int tiles = 1 + sa_expert_tiles_max(P, E, 16);   // (1 + ceil(P / 16) + min(E, P): as many experts as asked for)
  SA_REQUIRE(tiles <= kGridMax, "expert_product_shared: %d tiles", tiles);
  const dim3 grid(((N > shared_N ? N : shared_N) + 15) / 16, tiles);
  const SharedExpert sh{static_cast<const bf16*>(shared_h), static_cast<const bf16*>(shared_w), shared_y, shared_h_stride,
                        shared_y_stride, shared_N, shared_K, T};
  expert_product_kernel<bf16, false, 1, true><<<grid, kWave, 0, stream>>>(
      static_cast<const bf16*>(h), h_stride, 0, top, static_cast<const bf16*>(w), nullptr, N, K, sorted, plan, 0, 0.f, y, y_stride, 1, 0, sh);
  return check_launch("expert_product_shared");
}

extern "C" int sa_expert_product_beside_takes(int N, int K, int64_t h_stride, int P, int tile_rows, const void* shared_h,
                                              int64_t shared_h_stride, const void* shared_w, int shared_K, int T) {
  alignas(16) static const char aligned_stand_in[16] = {};   // (the experts' operands and the results are whole tensors)
  const void* p = aligned_stand_in;
  return N > 0 && K > 0 && P > 0 && T > 0 && shared_K > 0 && shared_h_stride >= shared_K &&
         gemm_wide_routed_takes(N, K, h_stride, P, N, p, p, nullptr, p, tile_rows) &&
         gemm_wide_routed_takes(N, shared_K, shared_h_stride, T, N, shared_h, shared_w, nullptr, p, tile_rows);
}

// Whether that launch is expected to be ahead of the experts' second products and a launch of the shared one's, with tiles of 128 rows.  The
// host counts what the CUs get: an expert's tokens as even routing deals them out, tile after tile to the CU that is free first, the
// shared product's behind the experts' (an XCD's workgroups start in the grid's order).  Rounds do not end as sharply as counted, so that it
// is taken up to 8 us behind.  Both second products and the experts' first, us, apart / beside, at expected gains in us: 16 experts of 2,048
// x 2,048, 2 chosen, shared of 2,048: 640 tokens 127 / 109 (15), 1,500 162 / 162 (-7), 2,047 209 / 185 (23); shared of 3,072: 774 132 / 118
// (7), 1,280 168 / 172 (-11), 2,047 218 / 196 (18); of 8,192: 774 166 / 177 (-34), 2,047 264 / 258 (-3), 4,096 401 / 382 (35); 4,096 x 3,584: 500
// 307 / 315 (-24), 1,024 409 / 378 (33); 64 experts, 8 chosen, 500 400 / 412 (-16); 8 experts of 4,096 x 3,584, one chosen, shared of
// 7,168: 774 239 / 207 (14), 3,000 471 / 514 (-56).  Of 116 sizes none is taken that is slower by 1.5 %.
extern "C" int sa_expert_product_beside_pays(int N, int K, int P, int E, int shared_K, int T) {
  if (N < 1 || K < 1 || P < 1 || E < 1 || shared_K < 1 || T < 1) return 0;
  constexpr int kRows = kTileRowsWide, kCUs = 256;
  const double mean = static_cast<double>(P) / E, deviation = sqrt(mean * (1.0 - 1.0 / E)) + 1e-9;
  double tiles = 0.0;   // of an expert: the sum over k of the chance that it has more than 128 k tokens
  for (int k = 0; k * kRows <= P; ++k) {
    const double more = 0.5 * erfc((k * kRows + 0.5 - mean) / (deviation * sqrt(2.0)));
    tiles += more;
    if (more < 1e-6 && k * kRows > mean) break;
  }
  const int columns = (N + 255) / 256;
  const int64_t own = llround(E * tiles * columns);
  int64_t left = static_cast<int64_t>((T + kRows - 1) / kRows) * columns;
  const double own_us = gemm_wide_tile_us(K), shared_us = gemm_wide_tile_us(shared_K);
  const double apart = (own + kCUs - 1) / kCUs * own_us +
                       fmin(gemm_wide_predict_us(T, N, shared_K, 0, true, size_t{256} << 20, false), gemm_tiled_predict_us(T, N, shared_K, 0));
  // the CUs that are free before the experts' last round and those behind it, each with the time from which they are
  double early = own / kCUs * own_us, late = early + own_us, beside = own % kCUs ? late : early;
  int64_t early_cus = kCUs - own % kCUs, late_cus = own % kCUs;
  while (left > 0) {
    const bool first = late_cus == 0 || early <= late;
    double& from = first ? early : late;
    left -= first ? early_cus : late_cus;
    from += shared_us;
    beside = fmax(beside, from);
  }
  return beside <= apart + 8.0;
}

extern "C" int sa_expert_product_beside(const void* h, int64_t h_stride, int top, const void* w, int N, int K, const int* sorted,
                                        const int* plan, int P, int E, int tile_rows, void* y, int64_t y_stride, const void* shared_h,
                                        int64_t shared_h_stride, const void* shared_w, int shared_K, int T, void* shared_y,
                                        int64_t shared_y_stride, hipStream_t stream) {
  SA_REQUIRE(P > 0 && E > 0 && N > 0 && K > 0 && top > 0 && T > 0 && shared_K > 0 && h_stride >= K && y_stride >= N &&
                 shared_h_stride >= shared_K && shared_y_stride >= N,
             "expert_product_beside: bad sizes P=%d E=%d N=%d K=%d T=%d K=%d", P, E, N, K, T, shared_K);
  SA_REQUIRE(h != nullptr && w != nullptr && sorted != nullptr && plan != nullptr && y != nullptr && shared_h != nullptr &&
                 shared_w != nullptr && shared_y != nullptr,
             "expert_product_beside: a null pointer");
  SA_REQUIRE(tile_rows == kTileRowsMax || tile_rows == kTileRowsWide, "expert_product_beside: tiles of %d or %d rows", kTileRowsMax, kTileRowsWide);
  const int tiles = sa_expert_tiles_max(P, E, tile_rows);
  SA_REQUIRE(static_cast<int64_t>(tiles) + (T + tile_rows - 1) / tile_rows <= kGridMax &&
                 gemm_wide_routed_takes(N, K, h_stride, P, y_stride, h, w, nullptr, y, tile_rows) &&
                 gemm_wide_routed_takes(N, shared_K, shared_h_stride, T, shared_y_stride, shared_h, shared_w, nullptr, shared_y, tile_rows),
             "expert_product_beside: aligned bfloat16 operands, K in multiples of 64; got N=%d K=%d and K=%d", N, K, shared_K);
  return gemm_wide_routed(h, h_stride, w, nullptr, nullptr, static_cast<float*>(y), y_stride, tiles, N, K, tile_rows, plan, sorted, 0, top, 0,
                          0.f, stream, shared_h, shared_h_stride, shared_w, shared_y, shared_y_stride, shared_K, T);
}

extern "C" int sa_expert_combine(const float* y, const float* weights, int top, const void* shared, int shared_dtype,
                                 int64_t shared_stride, const float* gate, int64_t gate_stride, void* out, int out_dtype,
                                 int64_t out_stride, int T, int D, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && T <= 65535 && D > 0 && top > 0 && out_stride >= D, "expert_combine: bad sizes T=%d D=%d top=%d", T, D,
             top);
  SA_REQUIRE(y != nullptr && weights != nullptr && out != nullptr, "expert_combine: a null pointer");
  SA_REQUIRE(shared == nullptr || shared_stride >= D, "expert_combine: the shared rows are too short");
  const auto aligned = [](const void* p, int64_t stride, int dtype) {
    return (reinterpret_cast<uintptr_t>(p) & (dtype == kF32 ? 15u : 7u)) == 0 && stride % 4 == 0;
  };
  if (D % 4 == 0 && aligned(y, 0, kF32) && (shared == nullptr || aligned(shared, shared_stride, shared_dtype)) &&
      aligned(out, out_stride, out_dtype) && (out_dtype == kF32 || out_dtype == kBF16) &&
      (shared == nullptr || shared_dtype == kF32 || shared_dtype == kBF16)) {
    const dim3 grid((D / 4 + 255) / 256, T);
#define SA_COMBINE(ST, OT)                                                                                           \
  combine_fours_kernel<ST, OT><<<grid, 256, 0, stream>>>(y, weights, top, static_cast<const ST*>(shared), shared_stride, gate, \
                                                         gate_stride, static_cast<OT*>(out), out_stride, D)
    const bool s32 = shared != nullptr && shared_dtype == kF32;
    if (s32 && out_dtype == kF32) SA_COMBINE(float, float);
    else if (s32) SA_COMBINE(float, bf16);
    else if (out_dtype == kF32) SA_COMBINE(bf16, float);
    else SA_COMBINE(bf16, bf16);
#undef SA_COMBINE
    return check_launch("expert_combine");
  }
  combine_kernel<<<dim3((D + 255) / 256, T), 256, 0, stream>>>(y, weights, top, shared, shared_dtype, shared_stride, gate,
                                                               gate_stride, out, out_dtype, out_stride, D);
  return check_launch("expert_combine");
}
