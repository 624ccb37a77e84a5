// Paged attention in 32 bits on the matrix cores (v_mfma_f32_16x16x4_f32, IEEE single precision), for head sizes of 64, 128
// and 256 in pages of a multiple of 16 keys; other sizes and options of the 32-bit path go to attention_generic.hip.
//
// A unit is up to 16 query rows (consecutive tokens of one request times the heads of a key head).  Its keys are taken in
// chunks of 64 aligned to absolute positions, a wave per chunk, four neighbouring chunks (a range of 256 keys) to a
// workgroup: scores S^T = K . Q^T, cap, mask, maximum, exponentials, O^T = V^T . P^T, all in the wave's registers, nothing
// exchanged between lanes but row maxima and sums (a 16 x 16 result holds rows 4 g + r, g = lane / 16, and column lane % 16;
// the products of a sum over k may take k in any order, so step r of the value product takes keys 4 g + r of both operands).
// A range's four chunks are added up through LDS, ranges one after the other.  The order of every sum is fixed by the
// query's position, so a token's result does not depend on how the tokens were cut into steps, on its unit, on what else is
// in the batch or on which pages hold the keys.  Three ways of running the ranges, with the same arithmetic (sa_paged_attention_f32_parts
// says which, and why):
//
//   a workgroup per unit, key head and chunk, four waves to it, partial results to the workspace, a merge kernel: few units and ranges,
//   whose chunks are all there is to fill the chip with;
//   a workgroup per unit, key head and range, partial results and a merge likewise: more of them, longer prompts;
//   a workgroup per unit and key head that walks through the ranges: many decoding requests, units of one or two tokens (more than four
//   heads a key head), and where the workspace holds no part for every range: an engine's 256 MiB hold those of a portion of 2,048
//   tokens of 8 heads over 4 key heads of 256, or of 1,024 tokens of 32 heads over 16 of 128, up to 3,840 keys.
//
// Keys that some row of the unit does not see get the weight zero.  Where such keys' values are not finite (a zero weight
// would spread them), their products are taken one key at a time and left out of the rows that do not see it.
//
// Scores are summed in a chain of products for each 32 entries of a head: results are 0.5 to 0.75 times as far from 64 bits as
// the generic kernel's at heads of 256 (1.06 to 1.3 times with two chains).
//
// Bound by the latency of a wave's chunk (loads of keys, scores, exponentials, values, one after the other) at the measured
// sizes, 2B heads: 4 requests of 257 to 1,023 keys 10.4 us and 5.4 for the merge, where the generic kernel, a workgroup per
// token and key head that walks through all keys on the vector ALU, took 786; a prompt of 509 tokens 35 us for 498 (42 walked).
#include "api.h"
#include "attention_common.h"

namespace sa {
namespace f32att {

constexpr int kChunkKeys = 64, kRangeKeys = 256, kWaves = kRangeKeys / kChunkKeys;
constexpr int kExtra = 4;   // a partial row's maximum and sum behind its values (rows stay 16-byte aligned)

struct Args {
  const float* q;
  const float* k_pages;
  const float* v_pages;
  const int* table;
  const SeqMeta* units;
  float* out;
  const float* sinks;
  int64_t q_stride, out_stride;
  int table_stride, Kh, G, page_size, window;
  float cap, scale;
};

__device__ __forceinline__ void unit_keys(const SeqMeta& u, int window, int* lo, int* hi) {
  *hi = u.pos0 + u.q_len;
  *lo = (window > 0 && u.pos0 - window + 1 > 0) ? u.pos0 - window + 1 : 0;
}

// The weight of a part whose maximum is m in a sum whose maximum is top (an empty part: nothing).
__device__ __forceinline__ float part_weight(float m, float top) { return m == -INFINITY ? 0.f : expf(m - top); }

// A row's running result: V neighbouring values of it in a thread.
template <int V>
struct Running {
  float m, l;
  floatx4 o[V / 4];
  __device__ __forceinline__ void clear() {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int i = 0; i < V / 4; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void add(float pm, float pl, const floatx4 (&po)[V / 4]) {
    const float top = fmaxf(m, pm), a = part_weight(m, top), b = part_weight(pm, top);
    l = fmaf(l, a, pl * b);
#pragma unroll
    for (int i = 0; i < V / 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[i][e] = fmaf(o[i][e], a, po[i][e] * b);
    m = top;
  }
  // thread: row `row` of the unit, values d0 .. d0 + V - 1
  __device__ __forceinline__ void write(const Args& a, const SeqMeta& u, int kh, int row, int hd, int d0) const {
    if (row >= u.q_len * a.G) return;
    const int head = kh * a.G + row % a.G;
    const float sum = a.sinks != nullptr ? l + expf(a.sinks[head] - m) : l;
    float* dst = a.out + static_cast<size_t>(u.q_start + row / a.G) * a.out_stride + static_cast<size_t>(head) * hd + d0;
#pragma unroll
    for (int i = 0; i < V / 4; ++i)
      *reinterpret_cast<floatx4*>(dst + 4 * i) = floatx4{o[i][0] / sum, o[i][1] / sum, o[i][2] / sum, o[i][3] / sum};
  }
};

// Adds a range's chunks up under their common maximum: chunk(w, ..) gives chunk w's maximum, sum and V values of a row.
template <int V, typename Chunk>
__device__ __forceinline__ void add_chunks(Chunk chunk, float* top_out, float* sum_out, floatx4 (&po)[V / 4]) {
  float m[kWaves], l[kWaves], top = -INFINITY, sum = 0.f;
  floatx4 x[kWaves][V / 4];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) chunk(w, &m[w], &l[w], x[w]);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) top = fmaxf(top, m[w]);
#pragma unroll
  for (int i = 0; i < V / 4; ++i) po[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const float f = part_weight(m[w], top);
    sum = fmaf(l[w], f, sum);
#pragma unroll
    for (int i = 0; i < V / 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) po[i][e] = fmaf(x[w][i][e], f, po[i][e]);
  }
  *top_out = top, *sum_out = sum;
}

// A workgroup per unit, key head and chunk, its partial result to parts [unit * Kh + kh][chunk of the grid][16][hd + kExtra].  Each of
// the four waves scores a quarter of the chunk's keys, hands the weights to the others through LDS, and multiplies all of them with
// a quarter of the values' entries: a wave issues 128 matrix instructions where the chunk has 512 and waits for memory twice, on four
// times as many CUs as ranges would have.  Every sum is that of attention_f32_kernel, in its order.  NB: head size / 32.
// 4 requests of 257 to 1,023 keys, 2B heads: 10.4 us and 5.4 for the merge; with a wave a chunk and a workgroup a range 27.6, with four
// waves a chunk and a workgroup a range 25.5.  Bound by the chain of waits.
template <int NB>
__global__ __launch_bounds__(256, 2) void attention_f32_parts_kernel(Args a, int unit_begin, float* __restrict__ parts) {
  constexpr int HD = NB * 32, NT = HD / 16, MINE = NT / 4, ROW = HD + 4;
  __shared__ __align__(16) float q_s[16 * ROW];
  __shared__ __align__(16) floatx4 p_s[4][kWave];
  __shared__ float m_p[4][16];
  __shared__ int odd_s;   // pieces with values that are not finite at keys that some row does not see
  const int tid = threadIdx.x, lane = tid % kWave, part = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int c = lane % 16, g = lane / 16, kh = blockIdx.y;
  const SeqMeta u = a.units[unit_begin + blockIdx.x];
  if (u.q_len <= 0) return;
  int lo, hi;
  unit_keys(u, a.window, &lo, &hi);
  const int c0 = lo / kRangeKeys * kRangeKeys + static_cast<int>(blockIdx.z) * kChunkKeys;
  if (c0 >= hi || c0 + kChunkKeys <= lo) return;
  const int* table = a.table + static_cast<size_t>(u.slot) * a.table_stride;
  if (tid == 0) odd_s = 0;
  const float* kp = nullptr;
  const float* vp[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {   // (a piece that no row sees stands for the nearest one that is seen)
    int key = c0 + 16 * s;
    key = key + 15 < lo ? lo / 16 * 16 : key >= hi ? (hi - 1) / 16 * 16 : key;
    const size_t page = static_cast<size_t>(table[key / a.page_size]) * a.Kh + kh;
    const int in_page = key % a.page_size;
    if (s == part) kp = a.k_pages + (page * a.page_size + in_page) * HD + lane * 8;   // (keys in blocks of 16 x 32, see common.h)
    vp[s] = a.v_pages + (page * HD + part * MINE * 16 + c) * a.page_size + in_page + 4 * g;
  }
  floatx4 k[NB][2], v[4][MINE];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 2; ++e) k[b][e] = *reinterpret_cast<const floatx4*>(kp + b * 512 + e * 4);
  // the unit's rows of queries (rows that are not there: the first)
  for (int i = tid; i < 16 * HD / 4; i += 256) {
    const int row = i / (HD / 4), d = i % (HD / 4) * 4;
    const bool there = row < u.q_len * a.G;
    const float* from = a.q + static_cast<size_t>(u.q_start + (there ? row / a.G : 0)) * a.q_stride +
                        static_cast<size_t>(kh * a.G + (there ? row % a.G : 0)) * HD + d;
    *reinterpret_cast<floatx4*>(&q_s[row * ROW + d]) = *reinterpret_cast<const floatx4*>(from);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int t = 0; t < MINE; ++t) v[s][t] = *reinterpret_cast<const floatx4*>(vp[s] + static_cast<size_t>(t) * 16 * a.page_size);
  const bool live = c < u.q_len * a.G;
  const int pos = u.pos0 + (live ? c / a.G : 0);
  const int row_lo = a.window > 0 ? pos - a.window : -1;   // keys behind this one are seen
  __syncthreads();
  floatx4 x[NB], p;
#pragma unroll
  for (int b = 0; b < NB; ++b) {   // (a chain for each 32 entries: a long one rounds at its size with every product)
    x[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    floatx4 q[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) q[e] = *reinterpret_cast<const floatx4*>(&q_s[c * ROW + b * 32 + g * 8 + e * 4]);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[b][e / 4][e % 4], q[e / 4][e % 4], x[b], 0, 0, 0);
  }
#pragma unroll
  for (int n = NB / 2; n > 0; n /= 2)
#pragma unroll
    for (int b = 0; b < n; ++b) x[b] += x[b + n];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int key = c0 + 16 * part + 4 * g + i;
    float y = x[0][i] * a.scale;
    if (a.cap > 0.f) y = a.cap * tanhf(y / a.cap);
    p[i] = key <= pos && key > row_lo ? y : -INFINITY;
  }
  const float mine = max_over_row_lanes(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3])));
  if (g == 0) m_p[part][c] = mine;
  __syncthreads();
  const float m = fmaxf(fmaxf(m_p[0][c], m_p[1][c]), fmaxf(m_p[2][c], m_p[3][c]));
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = p[i] == -INFINITY ? 0.f : expf(p[i] - m);   // (a row that sees nothing here: all zero)
  p_s[part][lane] = p;
  // values of keys that some row does not see
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int key = c0 + 16 * s;
    // every row of the unit sees the keys from its last row's first key to its first row's position
    const bool whole = key > u.pos0 + u.q_len - 1 - (a.window > 0 ? a.window : 0x3fffffff) && key + 15 <= u.pos0;
    if (key >= hi || key + 15 < lo || whole) continue;   // (uniform)
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = key + 4 * g + i;
      const bool held = at >= lo && at < hi;   // (what lies beyond has not been written, or is another's by now)
#pragma unroll
      for (int t = 0; t < MINE; ++t) {
        v[s][t][i] = held ? v[s][t][i] : 0.f;
        odd |= !(fabsf(v[s][t][i]) < INFINITY);
      }
    }
    if (__any(odd) && lane == 0) atomicOr(&odd_s, 1 << s);
  }
  __syncthreads();
  float l = 0.f;
  floatx4 o[MINE];
#pragma unroll
  for (int t = 0; t < MINE; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int odd = __builtin_amdgcn_readfirstlane(odd_s);
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const floatx4 w = p_s[s][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) l += w[i];
    const int key = c0 + 16 * s;
    if (key >= hi || key + 15 < lo) continue;   // (uniform)
    if ((odd >> s & 1) == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < MINE; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[s][t][i], w[i], o[t], 0, 0, 0);
    } else {
      for (int j = 0; j < 16; ++j) {
        const bool seen = key + j <= pos && key + j > row_lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (j % 4 != i) continue;
          const bool of_lane = j / 4 == g;
#pragma unroll
          for (int t = 0; t < MINE; ++t) {
            const floatx4 one = __builtin_amdgcn_mfma_f32_16x16x4f32(of_lane ? v[s][t][i] : 0.f, of_lane ? w[i] : 0.f,
                                                                     floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[t][e] += seen ? one[e] : 0.f;
          }
        }
      }
    }
  }
  l = sum_over_row_lanes(l);
  if (!live) return;
  float* dst = parts + ((static_cast<size_t>(blockIdx.x) * a.Kh + kh) * gridDim.z + blockIdx.z) * (16 * (HD + kExtra)) +
               static_cast<size_t>(c) * (HD + kExtra);
#pragma unroll
  for (int t = 0; t < MINE; ++t) *reinterpret_cast<floatx4*>(dst + (part * MINE + t) * 16 + g * 4) = o[t];
  if (g == 0 && part == 0) *reinterpret_cast<floatx4*>(dst + HD) = floatx4{m, l, 0.f, 0.f};
}

// A workgroup per unit and key head that walks through the ranges, a wave a chunk; or (PARTS) one for each range, its partial result
// to parts [unit * Kh + kh][range of the grid][16][hd + kExtra].  NB: head size / 32.
template <int NB, bool PARTS>
__global__ __launch_bounds__(256, NB == 8 && !PARTS ? 1 : 2) void attention_f32_kernel(Args a, int unit_begin, float* __restrict__ parts) {
  constexpr int HD = NB * 32, NT = HD / 16, V = HD / 16, ROW = HD + 4;
  __shared__ __align__(16) float o_s[kWaves][16 * ROW];
  __shared__ float m_s[kWaves][16], l_s[kWaves][16];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int c = lane % 16, g = lane / 16, kh = blockIdx.y;
  const SeqMeta u = a.units[unit_begin + blockIdx.x];
  if (u.q_len <= 0) return;
  int lo, hi;
  unit_keys(u, a.window, &lo, &hi);
  const int r0 = lo / kRangeKeys + (PARTS ? static_cast<int>(blockIdx.z) : 0);
  const int r1 = PARTS ? r0 + 1 : (hi + kRangeKeys - 1) / kRangeKeys;
  if (r0 * kRangeKeys >= hi) return;
  const int* table = a.table + static_cast<size_t>(u.slot) * a.table_stride;

  // the lane's row of queries: entries 32 b + 8 g .. + 7
  floatx4 q[NB][2];
  const bool live = c < u.q_len * a.G;
  {
    const int token = live ? c / a.G : 0, head = kh * a.G + (live ? c % a.G : 0);
    const float* qp = a.q + static_cast<size_t>(u.q_start + token) * a.q_stride + static_cast<size_t>(head) * HD + g * 8;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 2; ++e) q[b][e] = *reinterpret_cast<const floatx4*>(qp + b * 32 + e * 4);
  }
  const int pos = u.pos0 + (live ? c / a.G : 0);
  const int row_lo = a.window > 0 ? pos - a.window : -1;   // keys behind this one are seen

  const int row = tid / 16, d0 = tid % 16 * V;   // what the thread adds up
  Running<V> run;
  run.clear();
  for (int r = r0; r < r1; ++r) {
    const int c0 = r * kRangeKeys + wave * kChunkKeys;
    float m = -INFINITY, l = 0.f;
    floatx4 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (c0 < hi && c0 + kChunkKeys > lo) {   // (uniform over the wave)
      // pages of the chunk's four pieces of 16 keys; a piece that no row sees stands for the nearest one that is seen
      const float* kp[4];
      const float* vp[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        int key = c0 + 16 * s;
        key = key + 15 < lo ? lo / 16 * 16 : key >= hi ? (hi - 1) / 16 * 16 : key;
        const size_t page = static_cast<size_t>(table[key / a.page_size]) * a.Kh + kh;
        const int in_page = key % a.page_size;
        kp[s] = a.k_pages + (page * a.page_size + in_page) * HD + lane * 8;   // (keys in blocks of 16 x 32, see common.h)
        vp[s] = a.v_pages + (page * HD + c) * a.page_size + in_page + 4 * g;
      }
      floatx4 p[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        floatx4 k[NB][2], x[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 2; ++e) k[b][e] = *reinterpret_cast<const floatx4*>(kp[s] + b * 512 + e * 4);
#pragma unroll
        for (int b = 0; b < NB; ++b) {   // (a chain for each 32 entries: a long one rounds at its size with every product)
          x[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 8; ++e) x[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[b][e / 4][e % 4], q[b][e / 4][e % 4], x[b], 0, 0, 0);
        }
#pragma unroll
        for (int n = NB / 2; n > 0; n /= 2)
#pragma unroll
          for (int b = 0; b < n; ++b) x[b] += x[b + n];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = c0 + 16 * s + 4 * g + i;
          float v = x[0][i] * a.scale;
          if (a.cap > 0.f) v = a.cap * tanhf(v / a.cap);
          p[s][i] = key <= pos && key > row_lo ? v : -INFINITY;
          m = fmaxf(m, p[s][i]);
        }
      }
      m = max_over_row_lanes(m);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[s][i] = p[s][i] == -INFINITY ? 0.f : expf(p[s][i] - m);   // (a row that sees nothing here: all zero)
          l += p[s][i];
        }
      l = sum_over_row_lanes(l);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int key = c0 + 16 * s;
        if (key >= hi || key + 15 < lo) continue;   // (uniform)
        floatx4 v[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) v[t] = *reinterpret_cast<const floatx4*>(vp[s] + static_cast<size_t>(t) * 16 * a.page_size);
        // every row of the unit sees the keys from its last row's first key to its first row's position
        const bool whole = key > u.pos0 + u.q_len - 1 - (a.window > 0 ? a.window : 0x3fffffff) && key + 15 <= u.pos0;
        bool odd = false;
        if (!whole) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int at = key + 4 * g + i;
            const bool held = at >= lo && at < hi;   // (what lies beyond has not been written, or is another's by now)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              v[t][i] = held ? v[t][i] : 0.f;
              odd |= !(fabsf(v[t][i]) < INFINITY);
            }
          }
          odd = __any(odd);
        }
        if (!odd) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][i], p[s][i], o[t], 0, 0, 0);
        } else {
          for (int j = 0; j < 16; ++j) {
            const bool seen = key + j <= pos && key + j > row_lo;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              if (j % 4 != i) continue;
              const bool mine = j / 4 == g;
#pragma unroll
              for (int t = 0; t < NT; ++t) {
                const floatx4 one = __builtin_amdgcn_mfma_f32_16x16x4f32(mine ? v[t][i] : 0.f, mine ? p[s][i] : 0.f,
                                                                         floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[t][e] += seen ? one[e] : 0.f;
              }
            }
          }
        }
      }
    }
    if (r > r0) __syncthreads();   // (the range before has been added up)
#pragma unroll
    for (int t = 0; t < NT; ++t) *reinterpret_cast<floatx4*>(&o_s[wave][c * ROW + t * 16 + g * 4]) = o[t];
    if (g == 0) {
      m_s[wave][c] = m;
      l_s[wave][c] = l;
    }
    __syncthreads();
    float top, sum;
    floatx4 po[V / 4];
    add_chunks<V>([&](int w, float* cm, float* cl, floatx4 (&x)[V / 4]) __attribute__((always_inline)) {
      *cm = m_s[w][row], *cl = l_s[w][row];
#pragma unroll
      for (int i = 0; i < V / 4; ++i) x[i] = *reinterpret_cast<const floatx4*>(&o_s[w][row * ROW + d0 + 4 * i]);
    }, &top, &sum, po);
    if constexpr (PARTS) {
      float* dst = parts + ((static_cast<size_t>(blockIdx.x) * a.Kh + kh) * gridDim.z + blockIdx.z) * (16 * (HD + kExtra)) +
                   static_cast<size_t>(row) * (HD + kExtra);
#pragma unroll
      for (int i = 0; i < V / 4; ++i) *reinterpret_cast<floatx4*>(dst + d0 + 4 * i) = po[i];
      if (tid % 16 == 0) *reinterpret_cast<floatx4*>(dst + HD) = floatx4{top, sum, 0.f, 0.f};
    } else {
      run.add(top, sum, po);
    }
  }
  if constexpr (!PARTS) run.write(a, u, kh, row, HD, d0);
}

// A unit's ranges: sixteen threads for a row, with V values each on their way at once (one request of 65,536 keys, 2B heads, 221 us with
// its attention; 242 with four values a thread, as below).
template <int NB>
__global__ __launch_bounds__(256) void attention_f32_merge_kernel(Args a, int unit_begin, const float* __restrict__ parts, int ranges) {
  constexpr int HD = NB * 32, V = HD / 16;
  const SeqMeta u = a.units[unit_begin + blockIdx.x];
  if (u.q_len <= 0) return;
  int lo, hi;
  unit_keys(u, a.window, &lo, &hi);
  const int kh = blockIdx.y, row = threadIdx.x / 16, d0 = threadIdx.x % 16 * V;
  const int n = (hi + kRangeKeys - 1) / kRangeKeys - lo / kRangeKeys;
  const float* src = parts + (static_cast<size_t>(blockIdx.x) * a.Kh + kh) * ranges * (16 * (HD + kExtra)) +
                     static_cast<size_t>(row) * (HD + kExtra);
  Running<V> run;
  run.clear();
  for (int z = 0; z < n && z < ranges; ++z, src += 16 * (HD + kExtra)) {
    floatx4 po[V / 4];
#pragma unroll
    for (int i = 0; i < V / 4; ++i) po[i] = *reinterpret_cast<const floatx4*>(src + d0 + 4 * i);
    run.add(src[HD], src[HD + 1], po);
  }
  run.write(a, u, kh, row, HD, d0);
}

// A unit's chunks, by ranges: four neighbouring values of a row in a thread, threads for the rows of the longest unit.
template <int NB>
__global__ __launch_bounds__(4 * NB * 32) void attention_f32_merge_chunks_kernel(Args a, int unit_begin, const float* __restrict__ parts, int ranges) {
  constexpr int HD = NB * 32;
  const SeqMeta u = a.units[unit_begin + blockIdx.x];
  const int kh = blockIdx.y, row = threadIdx.x / (HD / 4), d0 = threadIdx.x % (HD / 4) * 4;
  if (row >= u.q_len * a.G) return;
  int lo, hi;
  unit_keys(u, a.window, &lo, &hi);
  const int first = lo / kRangeKeys, n = (hi + kRangeKeys - 1) / kRangeKeys - first;
  const float* src = parts + (static_cast<size_t>(blockIdx.x) * a.Kh + kh) * ranges * kWaves * (16 * (HD + kExtra)) +
                     static_cast<size_t>(row) * (HD + kExtra);
  Running<4> run;
  run.clear();
  for (int z = 0; z < n && z < ranges; ++z) {
    float top, sum;
    floatx4 po[1];
    add_chunks<4>([&](int w, float* cm, float* cl, floatx4 (&x)[1]) __attribute__((always_inline)) {
      const int c0 = (first + z) * kRangeKeys + w * kChunkKeys;
      const float* from = src + static_cast<size_t>(z * kWaves + w) * (16 * (HD + kExtra));
      const bool there = c0 < hi && c0 + kChunkKeys > lo;   // (others have written nothing: what lies there is read and not used)
      const floatx4 ml = *reinterpret_cast<const floatx4*>(from + HD), y = *reinterpret_cast<const floatx4*>(from + d0);
      *cm = there ? ml[0] : -INFINITY, *cl = there ? ml[1] : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[0][e] = there ? y[e] : 0.f;
    }, &top, &sum, po);
    run.add(top, sum, po);
  }
  run.write(a, u, kh, row, HD, d0);
}

template <int NB>
static void launch(const Args& a, int unit_begin, int units, int rows, int ranges, int per, float* parts, hipStream_t stream) {
  if (per == kWaves) {
    attention_f32_parts_kernel<NB><<<dim3(units, a.Kh, ranges * kWaves), 256, 0, stream>>>(a, unit_begin, parts);
    attention_f32_merge_chunks_kernel<NB><<<dim3(units, a.Kh), rows * NB * 8, 0, stream>>>(a, unit_begin, parts, ranges);
  } else if (per == 1) {
    attention_f32_kernel<NB, true><<<dim3(units, a.Kh, ranges), 256, 0, stream>>>(a, unit_begin, parts);
    attention_f32_merge_kernel<NB><<<dim3(units, a.Kh), 256, 0, stream>>>(a, unit_begin, parts, ranges);
  } else {
    attention_f32_kernel<NB, false><<<dim3(units, a.Kh), 256, 0, stream>>>(a, unit_begin, nullptr);
  }
}

}  // namespace f32att
}  // namespace sa

using namespace sa;

extern "C" int sa_paged_attention_f32_takes(int H, int Kh, int hd, int page_size, int64_t q_stride, const void* q) {
  return Kh > 0 && Kh <= 65535 && H % Kh == 0 && H / Kh <= 16 && (hd == 64 || hd == 128 || hd == 256) && page_size > 0 &&
         page_size % 16 == 0 && q_stride % 4 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0;
}

// Ranges that a unit's keys can touch.
static int f32_ranges(int window, int max_kv_len, int max_q_len) {
  const int64_t seen = window > 0 && static_cast<int64_t>(window) + max_q_len - 1 < max_kv_len ? static_cast<int64_t>(window) + max_q_len - 1 : max_kv_len;
  return static_cast<int>(seen < max_kv_len ? (seen + f32att::kRangeKeys - 2) / f32att::kRangeKeys + 1
                                            : (seen + f32att::kRangeKeys - 1) / f32att::kRangeKeys);
}

extern "C" int sa_paged_attention_f32_parts(int unit_count, int Kh, int hd, int window, int max_kv_len, int max_q_len, int64_t workspace_bytes) {
  const int ranges = f32_ranges(window, max_kv_len, max_q_len);
  const int64_t heads = static_cast<int64_t>(unit_count) * Kh;
  const int64_t bytes = heads * ranges * 16 * (hd + f32att::kExtra) * static_cast<int64_t>(sizeof(float));   // a part a range
  // Prompts (units of four tokens and more; up to four heads a key head have such, prompts of more walk as before): a unit sees what lies
  // before it, so units that walk are as slow as the last one's ranges one after the other, and a chunk is a chain of waits of 10 us that
  // more workgroups cover.  What the workspace does not hold walks.  Walked / ranges / chunks in us, heads of 256,
  // 4 key heads, by triples (see below): 64 tokens (32) 20 / 20 / 12, behind 2,048 others (288) 186 / 43 / 44; 509 (512) 42 / 38 / 35; 700
  // (1,056) 83 / 62 / 51; behind 512 (1,760) 163 / 97 / 96; 384 behind 2,048 (1,920) 198 / 125 / 124; 1,024 (2,048) 137 / 94 / 95; 509
  // behind 2,048 (2,560) 198 / 154 / 166; 2,048 (8,192) 397 / 274.  16 key heads of 128: 256 (512, one range) 20 / 23 / 25, 512 (2,048)
  // 62 / 52 / 59; 4 of 64: 128 (32) 8.6 / 10.5 / 7.3, 512 (256) 15.3 / 11.3 / 11.4, 16 heads over 4, 1,024 (4,096) 64 / 48 / 58.
  // A chunk's part is one more for the merge to walk through, so chunks end at six ranges (ranges / chunks: 17 tokens behind 8,000 (384)
  // 56 / 78, 5 behind 30,000 (472) 96 / 161, 100 behind 2,000 (468) 45 / 52; 64 behind 700 (96) 29 / 23), but where the ranges leave half
  // of the CUs idle (as below; up to 24 ranges: 118 of 2 tokens over one key head 74 / 150).  Over 1,528 sizes what is chosen takes
  // 1.5 % more than the best way, 20 % at worst: walking, of heads of 64 and 128 whose units all see two ranges and make whole rounds.
  if (max_q_len >= 4) {
    const int64_t triples = heads * ranges;
    if (((triples * 36 <= static_cast<int64_t>(hd) * hd && ranges <= 6) || (triples <= 128 && ranges <= 24)) &&
        bytes * f32att::kWaves <= workspace_bytes)
      return f32att::kWaves;
    return ranges > 1 && ranges <= 65535 && bytes <= workspace_bytes ? 1 : 0;
  }
  // Parts while the units alone do not fill the 256 CUs.
  if (ranges <= 1 || ranges > 65535 || heads >= 256 || bytes > workspace_bytes) return 0;
  // A workgroup per chunk while the ranges leave half of the CUs idle: beyond that, four times the parts cost the merge more than four
  // times the workgroups give.  Chunks / ranges in us, heads of 256, 4 key heads, by (unit, key head, range) triples: 64 (one request of
  // 4,096 keys) 21 / 30, 128 (one of 8,192) 38.5 / 39.8, (8 of 1,024) 21 / 28, 256 (one of 16,384) 66 / 58, (8 of 2,048) 34 / 34.5,
  // 512 (one of 32,768) 146 / 104, (16 of 2,048) 55 / 55; 16 key heads of 128: 64 (one of 1,024) 9.4 / 13.6, 256 (one of 4,096) 28 / 25.
  return heads * ranges <= 128 && bytes * f32att::kWaves <= workspace_bytes ? f32att::kWaves : 1;
}

extern "C" int sa_paged_attention_f32(const float* q, int64_t q_stride, const float* k_pages, const float* v_pages,
                                      const int* block_table, int table_stride, const int* units, int unit_begin,
                                      int unit_count, float* out, int64_t out_stride, int H, int Kh, int hd, int page_size,
                                      int window, float soft_cap, float scale, const float* sinks, int max_kv_len,
                                      int max_q_len, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  if (unit_count == 0) return 0;
  SA_REQUIRE(q != nullptr && k_pages != nullptr && v_pages != nullptr && block_table != nullptr && units != nullptr && out != nullptr,
             "paged_attention_f32: a null pointer");
  SA_REQUIRE(sa_paged_attention_f32_takes(H, Kh, hd, page_size, q_stride, q),
             "paged_attention_f32: does not take %d heads over %d of size %d, pages of %d", H, Kh, hd, page_size);
  SA_REQUIRE(unit_begin >= 0 && unit_count > 0 && table_stride > 0 && window >= 0 && max_kv_len > 0 && max_q_len > 0 &&
                 max_q_len * (H / Kh) <= 16,
             "paged_attention_f32: bad sizes: %d units of up to %d tokens, %d heads a key head", unit_count, max_q_len, H / Kh);
  SA_REQUIRE(q_stride >= static_cast<int64_t>(H) * hd && out_stride >= static_cast<int64_t>(H) * hd && out_stride % 4 == 0 &&
                 reinterpret_cast<uintptr_t>(out) % 16 == 0 && reinterpret_cast<uintptr_t>(k_pages) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(v_pages) % 16 == 0,
             "paged_attention_f32: rows too short or not aligned");
  f32att::Args a;
  a.q = q, a.k_pages = k_pages, a.v_pages = v_pages, a.table = block_table, a.units = reinterpret_cast<const SeqMeta*>(units);
  a.out = out, a.sinks = sinks, a.q_stride = q_stride, a.out_stride = out_stride, a.table_stride = table_stride, a.Kh = Kh;
  a.G = H / Kh, a.page_size = page_size, a.window = window, a.cap = soft_cap, a.scale = scale;
  const int ranges = f32_ranges(window, max_kv_len, max_q_len);
  const int per = workspace != nullptr ? sa_paged_attention_f32_parts(unit_count, Kh, hd, window, max_kv_len, max_q_len, workspace_bytes) : 0;
  float* parts = static_cast<float*>(workspace);
  if (hd == 64) f32att::launch<2>(a, unit_begin, unit_count, max_q_len * a.G, ranges, per, parts, stream);
  else if (hd == 128) f32att::launch<4>(a, unit_begin, unit_count, max_q_len * a.G, ranges, per, parts, stream);
  else f32att::launch<8>(a, unit_begin, unit_count, max_q_len * a.G, ranges, per, parts, stream);
  return check_launch("paged_attention_f32");
}
