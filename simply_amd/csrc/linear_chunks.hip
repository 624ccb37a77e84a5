// The recurrence of linear_state.hip with a decay per key channel, for portions of prompts of bfloat16 runs, on the matrix
// cores: 64 tokens (a piece) at a time.  With S the state in front of a piece and D_(a..b) the product of the decays of
// tokens a .. b, channel by channel,
//
//   o_i = (D_(1..i-1) q_i)^T S + sum_(j < i) M_ij v_j + ((bonus q_i) . k_i) v_i,   M_ij = sum_d q_i k_j D_(j+1..i-1)
//   S  <- D_(1..64) S + sum_j (D_(j+1..64) k_j) v_j^T
//
// (without a bonus a token reads the state behind it: D_(1..i), M_ij with D_(j+1..i) and M_ii = q_i . k_i).  No logarithms
// and no quotients of decays: products of decays between two tokens are taken as such, so that a decay of zero, or many
// small ones, do no harm.  Within a block of 16 tokens a lane holds a key and carries it from token to token, multiplied by
// their decays (16 lanes: the block's tokens; four groups of lanes: channels 16 n + 4 g + r); what it has become at the
// block's end is what later blocks see of it, and a query multiplied by the decays in front of it in its block, then by whole
// blocks', meets those keys in matrix products.
//
//   linear_pieces_kernel   everything that does not need the state, a workgroup per piece and head: M and the scaled queries,
//                          keys and values, in the order in which the second kernel's instructions take them
//   linear_walk_kernel     the walk through the pieces, a workgroup of four waves per head and 16 value columns, as
//                          delta_state_kernel does it (delta_chunks.hip), with one barrier a piece; or, for long requests of few
//                          heads (keeps_states), linear_scan_kernel for the state alone and piece_outputs_kernel, the same sums
//
// Sums and products are 32-bit (v_mfma_f32_16x16x4_f32).  The first kernel is bound by a wave's vector instructions (two
// times 16 steps of 32 multiplications in 64 bits with their conversions, of keys and of queries one after the other: with both
// at once a CU has registers for half the waves, 60 us instead of 46), the second by its matrix instructions one after the other.
//
// What keeps the error against 64 bits no larger than that of linear_state.hip: decays are multiplied in 64 bits, before they
// meet a key or query that is rounded once; sums run in chains of 16 products, the state's increment by itself; and over
// tokens step r of an operand takes tokens 4 r + g, so that a chain adds them in their order, whose last are the largest where
// decays are fast.  Times the error of linear_state.hip, results and state (80 to 260 tokens, 16 heads of 128):
//   rates per channel, decays 0.998 to 0.19       0.87 to 0.69   0.65 to 0.51
//   sigmoid(z)^(1 / 16)                           0.97           0.89 to 0.97
//   decays drawn anew for each token, 0.69 on     1.00           0.97 to 1.05
//   the same between 0 and 1                      0.96           1.25 to 1.40
// (with decays multiplied in 32 bits and two or four chains the second to fourth were 1.04 to 1.19 and 1.16 to 1.8.)
//
// Measured at 2,048 tokens of 16 heads of 128: 91 us (traced, 48 for the pieces, 22 for the scan and 25 for the outputs; 126 with the
// walk's 81 instead), where
// linear_state.hip takes 704 token by token.
#include "api.h"
#include "chunks.h"

namespace sa {
namespace linear {

using namespace chunks;

// A piece's operands in the workspace (floats), for NT blocks of 16 key channels and CB blocks of 16 value columns.
struct Layout {
  int q, kt, p, v, all, states, words;   // states: in front of the pieces, where they are kept
};
__host__ __device__ constexpr Layout layout(int nt, int cb, bool keep) {
  Layout l{};
  l.q = 0;                              // [token block][channel block]
  l.kt = l.q + kBlocks * nt * kBlock;   // [channel block][token block]
  l.p = l.kt + kBlocks * nt * kBlock;   // [token block][token block]
  l.v = l.p + kBlocks * kBlocks * kBlock;   // [column block][token block]
  l.all = l.v + cb * kBlocks * kBlock;      // [16 nt] the decays of the whole piece
  l.states = l.all + 16 * nt;               // [column block][channel block]
  l.words = l.states + (keep ? cb * nt * kBlock : 0);
  return l;
}

struct Args {
  const bf16* proj;
  const float* gates;   // [T, >= H dk]: decays, or z where inv_tau > 0
  const void* gate_bias;
  const void* bonus;
  float* state;         // per slot and head [dv][dk]
  float* out;           // [T, H * dv]
  float* pieces;
  const int* seq_meta;
  int64_t proj_stride, gates_stride, state_stride;
  float q_mult, inv_tau;
  int q_at, k_at, v_at, H, dk, dv, bias_dtype, bonus_dtype, row0, row1;
  bool keep;            // the states in front of the pieces
};

__device__ __forceinline__ floatx4 to_float4(uint2 v) {   // four bfloat16
  return floatx4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                 __uint_as_float(v.y & 0xffff0000u)};
}

template <int NT, bool BONUS>
__global__ __launch_bounds__(256) void linear_pieces_kernel(Args a) {
  constexpr int QUADS = NT * 4, AROW = NT * 16 + 4, QROW = NT * 16 + 8;
  __shared__ __align__(16) float a_s[kTokens * AROW];   // decays; then the keys as later blocks see them, [block][channel block][lane]
  __shared__ __align__(16) bf16 q_s[kTokens * QROW];
  __shared__ __align__(16) bf16 k_s[kTokens * QROW];
  __shared__ __align__(16) float blk_s[kBlocks][NT * 16];   // a block's decays, multiplied
  const Span sp = span_of(a.seq_meta, a.row0, a.row1, blockIdx.z);
  const int t0 = blockIdx.y * kTokens;
  if (t0 >= sp.count) return;   // (uniform)
  const int left = sp.count - t0 < kTokens ? sp.count - t0 : kTokens;
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), c = lane % 16, g = lane / 16;
  const int row0 = sp.first + t0, cb = (a.dv + 15) / 16;
  const Layout lay = layout(NT, cb, a.keep);
  float* dst = a.pieces + (static_cast<size_t>(sp.piece0 + blockIdx.y) * a.H + h) * lay.words;

  // rows of q, k and the decays (tokens behind the last: nothing, decays of one; channels behind the last: zeros)
#pragma unroll
  for (int i = 0; i < kTokens * QUADS / 256; ++i) {
    const int idx = tid + i * 256, j = idx / QUADS, d = idx % QUADS * 4;
    const bool ok = j < left && d < a.dk;
    uint2 qv{0, 0}, kv{0, 0};
    floatx4 av{1.f, 1.f, 1.f, 1.f};
    if (ok) {
      const bf16* row = a.proj + static_cast<size_t>(row0 + j) * a.proj_stride + h * a.dk + d;
      qv = *reinterpret_cast<const uint2*>(row + a.q_at);
      kv = *reinterpret_cast<const uint2*>(row + a.k_at);
      av = *reinterpret_cast<const floatx4*>(a.gates + static_cast<size_t>(row0 + j) * a.gates_stride + h * a.dk + d);
      if (a.inv_tau > 0.f) {   // a = sigmoid(z + bias)^(1 / tau)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float z = av[e] + (a.gate_bias != nullptr ? load_f(a.gate_bias, a.bias_dtype, h * a.dk + d + e) : 0.f);
          av[e] = __expf((fminf(z, 0.f) - __logf(1.f + __expf(-fabsf(z)))) * a.inv_tau);
        }
      }
    }
    *reinterpret_cast<uint2*>(&q_s[j * QROW + d]) = qv;
    *reinterpret_cast<uint2*>(&k_s[j * QROW + d]) = kv;
    *reinterpret_cast<floatx4*>(&a_s[j * AROW + d]) = av;
  }
  __syncthreads();
  // values of the wave's tokens, as the right operand: this lane has tokens 4 r + g
  for (int n = 0; n < cb; ++n) {
    const int col = n * 16 + c;
    floatx4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = wave * 16 + r * 4 + g;
      v[r] = j < left && col < a.dv ? to_float(a.proj[static_cast<size_t>(row0 + j) * a.proj_stride + a.v_at + h * a.dv + col]) : 0.f;
    }
    *reinterpret_cast<floatx4*>(dst + lay.v + (n * kBlocks + wave) * kBlock + lane * 4) = v;
  }
  // the block of 16 tokens on the diagonal: lane c has key c, and step i brings token i's decays and its query to all lanes' keys
  // (kw, times the decays behind the token so far, which are multiplied in 64 bits: a key that has been rounded 15 times over
  // would be the largest part of the results' error)
  double kw[NT][4];
  floatx4 own_r{0.f, 0.f, 0.f, 0.f};   // M_cc, by the lane's channels
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const floatx4 q = to_float4(*reinterpret_cast<const uint2*>(&q_s[(wave * 16 + c) * QROW + n * 16 + g * 4])) * a.q_mult;
    const floatx4 k = to_float4(*reinterpret_cast<const uint2*>(&k_s[(wave * 16 + c) * QROW + n * 16 + g * 4]));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = q[r] * k[r];
      const int d = n * 16 + g * 4 + r;
      if (BONUS) x *= d < a.dk ? load_f(a.bonus, a.bonus_dtype, static_cast<size_t>(h) * a.dk + d) : 0.f;
      own_r[r] += x;
      kw[n][r] = static_cast<double>(k[r]);
    }
  }
  const float own = sum_over_row_lanes((own_r[0] + own_r[1]) + (own_r[2] + own_r[3]));
  float m_c[4] = {0.f, 0.f, 0.f, 0.f};   // M[query 4 g + r][key c] of the block
  auto decay_of = [&](int i, int n) __attribute__((always_inline)) {   // token i's decays of the lane's channels of block n
    return *reinterpret_cast<const floatx4*>(&a_s[(wave * 16 + i) * AROW + n * 16 + g * 4]);
  };
#pragma unroll 1
  for (int i4 = 0; i4 < 4; ++i4) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = i4 * 4 + e;
      floatx4 av[NT], s_r{0.f, 0.f, 0.f, 0.f};
      const bf16* qi = &q_s[(wave * 16 + i) * QROW + g * 4];
#pragma unroll
      for (int n = 0; n < NT; ++n) av[n] = decay_of(i, n);
      auto decay_keys = [&]() __attribute__((always_inline)) {
        if (c < i) {
#pragma unroll
          for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) kw[n][r] *= static_cast<double>(av[n][r]);
        }
      };
      if (!BONUS) decay_keys();
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const floatx4 q = to_float4(*reinterpret_cast<const uint2*>(qi + n * 16));
#pragma unroll
        for (int r = 0; r < 4; ++r) s_r[r] = fmaf(q[r], static_cast<float>(kw[n][r]), s_r[r]);
      }
      if (BONUS) decay_keys();
      float s = sum_over_row_lanes((s_r[0] + s_r[1]) + (s_r[2] + s_r[3])) * a.q_mult;
      s = c < i ? s : c == i ? own : 0.f;
      if (g == i4) m_c[e] = s;
    }
  }
  floatx4 key[NT], qp[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) key[n][r] = static_cast<float>(kw[n][r]);
  // query c times the decays in front of it in the block, likewise
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    double x[4] = {1.0, 1.0, 1.0, 1.0};
#pragma unroll 4
    for (int i = 0; i < 16; ++i) {
      const floatx4 av = decay_of(i, n);
      if (BONUS ? i < c : i <= c) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] *= static_cast<double>(av[r]);
      }
    }
    const floatx4 q = to_float4(*reinterpret_cast<const uint2*>(&q_s[(wave * 16 + c) * QROW + n * 16 + g * 4])) * a.q_mult;
#pragma unroll
    for (int r = 0; r < 4; ++r) qp[n][r] = static_cast<float>(x[r] * static_cast<double>(q[r]));
  }
  // the block's M, turned: as the left operand lane (query c, group g) has keys 4 r + g
  {
    float* to = dst + lay.p + (wave * kBlocks + wave) * kBlock + (c % 4) * 64 + c / 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) to[(g * 4 + e) * 4] = m_c[e];
  }
  // the block's decays, channel by channel (in 64 bits: 15 roundings of a factor that all of a channel's sums have in common
  // would be the largest part of their error)
#pragma unroll
  for (int d = lane; d < NT * 16; d += kWave) {
    double x = 1.0;
#pragma unroll
    for (int j = 0; j < 16; ++j) x *= static_cast<double>(a_s[(wave * 16 + j) * AROW + d]);
    blk_s[wave][d] = static_cast<float>(x);
  }
  __syncthreads();   // (the decays have been read)
  floatx4* key_s = reinterpret_cast<floatx4*>(a_s);
  static_assert(kBlocks * NT * kWave * 16 <= kTokens * AROW * 4, "the keys lie where the decays lay");
#pragma unroll
  for (int n = 0; n < NT; ++n) key_s[(wave * NT + n) * kWave + lane] = key[n];
  __syncthreads();
  // keys of earlier blocks, from the nearest on; the queries take a block's decays on the way
#pragma unroll 1
  for (int b = wave - 1; b >= 0; --b) {
    // (the keys' rows are permuted so that the result's are the left operand's tokens: this lane has keys 4 r + g of query c)
    floatx4 x[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) x[n] = halves4(key_s[(b * NT + n) * kWave + g * 16 + (c % 4) * 4 + c / 4], qp[n]);
    *reinterpret_cast<floatx4*>(dst + lay.p + (wave * kBlocks + b) * kBlock + lane * 4) = sum_of(x);
#pragma unroll
    for (int n = 0; n < NT; ++n) qp[n] *= *reinterpret_cast<const floatx4*>(&blk_s[b][n * 16 + g * 4]);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) *reinterpret_cast<floatx4*>(dst + lay.q + (wave * NT + n) * kBlock + lane * 4) = qp[n];
  // the wave's keys times the decays of the blocks behind, turned: [channel c][tokens 4 r + g]
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    float f = 1.f;
    for (int b = wave + 1; b < kBlocks; ++b) f *= blk_s[b][n * 16 + c];
    floatx4 kt;
#pragma unroll
    for (int r = 0; r < 4; ++r) kt[r] = a_s[((wave * NT + n) * kWave + (c / 4) * 16 + r * 4 + g) * 4 + c % 4] * f;
    *reinterpret_cast<floatx4*>(dst + lay.kt + (n * kBlocks + wave) * kBlock + lane * 4) = kt;
  }
  if (tid < NT * 16) dst[lay.all + tid] = blk_s[0][tid] * blk_s[1][tid] * blk_s[2][tid] * blk_s[3][tid];
}

template <int NT>
__global__ __launch_bounds__(256) void linear_walk_kernel(Args a) {
  constexpr int NW = NT / 4;   // blocks of key channels whose state a wave holds
  __shared__ __align__(16) floatx4 s_s[2][NT * kWave];
  const Span sp = span_of(a.seq_meta, a.row0, a.row1, blockIdx.z);
  if (sp.count <= 0) return;
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), c = lane % 16, g = lane / 16;
  const int col = blockIdx.y * 16 + c;
  const bool col_ok = col < a.dv;
  const Layout lay = layout(NT, (a.dv + 15) / 16, a.keep);
  const float* src = a.pieces + (static_cast<size_t>(sp.piece0) * a.H + h) * lay.words;
  const size_t step = static_cast<size_t>(a.H) * lay.words;
  float* S = a.state + static_cast<size_t>(sp.slot) * a.state_stride + static_cast<size_t>(h) * a.dk * a.dv;
  floatx4 s[NW];
#pragma unroll
  for (int n = 0; n < NW; ++n) {
    const int d = (wave * NW + n) * 16 + g * 4;
    s[n] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (col_ok && d < a.dk) s[n] = *reinterpret_cast<const floatx4*>(S + static_cast<size_t>(col) * a.dk + d);
    s_s[0][(wave * NW + n) * kWave + lane] = s[n];
  }
  // a piece's operands, asked for a piece ahead
  floatx4 q[NT], kt[NW][kBlocks], p[kBlocks], v[kBlocks], v_own, all[NW];   // (p: blocks in front of the wave's own, and that)
  auto fetch_state = [&](const float* from) __attribute__((always_inline)) {   // what the state behind the piece needs
#pragma unroll
    for (int n = 0; n < NW; ++n) {
      all[n] = *reinterpret_cast<const floatx4*>(from + lay.all + (wave * NW + n) * 16 + g * 4);
#pragma unroll
      for (int b = 0; b < kBlocks; ++b)
        kt[n][b] = *reinterpret_cast<const floatx4*>(from + lay.kt + ((wave * NW + n) * kBlocks + b) * kBlock + lane * 4);
    }
  };
  auto fetch_rest = [&](const float* from) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NT; ++n) q[n] = *reinterpret_cast<const floatx4*>(from + lay.q + (wave * NT + n) * kBlock + lane * 4);
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
      v[b] = *reinterpret_cast<const floatx4*>(from + lay.v + (blockIdx.y * kBlocks + b) * kBlock + lane * 4);
      const int at = b < wave ? b : wave;   // (the last: the wave's own; others behind it: that again, not used)
      p[b] = *reinterpret_cast<const floatx4*>(from + lay.p + (wave * kBlocks + at) * kBlock + lane * 4);
    }
    v_own = *reinterpret_cast<const floatx4*>(from + lay.v + (blockIdx.y * kBlocks + wave) * kBlock + lane * 4);
  };
  fetch_state(src);
  fetch_rest(src);
  int now = 0;
  for (int t0 = 0; t0 < sp.count; t0 += kTokens, now ^= 1) {
    const float* next = t0 + kTokens < sp.count ? src + step : src;   // (behind the last piece: that one again, for nothing)
    __syncthreads();   // the state in front of the piece is there
    floatx4 st[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) st[n] = s_s[now][n * kWave + lane];
    // the state behind the piece, for the others to read
    // (summed by itself, a chain for each 16 tokens: 64 products added to the state one by one would round it 64 times)
#pragma unroll
    for (int n = 0; n < NW; ++n) {
      floatx4 more[kBlocks];
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) more[b] = mul4(kt[n][b], v[b], floatx4{0.f, 0.f, 0.f, 0.f});
      const floatx4 added = ((more[0] + more[1]) + more[2]) + more[3];
#pragma unroll
      for (int r = 0; r < 4; ++r) s[n][r] = fmaf(s[n][r], all[n][r], added[r]);
    }
#pragma unroll
    for (int n = 0; n < NW; ++n) s_s[now ^ 1][(wave * NW + n) * kWave + lane] = s[n];
    fetch_state(next);
    floatx4 o[NT], o2[kBlocks];
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) o2[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < NT; ++n) o[n] = mul4(q[n], st[n], floatx4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int b = 0; b < kBlocks - 1; ++b)
      if (b < wave) o2[b] = mul4(p[b], v[b], o2[b]);   // (uniform over the wave)
    o2[kBlocks - 1] = lower_mul4<true>(p[kBlocks - 1], v_own, o2[kBlocks - 1], lane);
    const floatx4 result = sum_of(o) + sum_of(o2);
    fetch_rest(next);
    if (col_ok) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + wave * 16 + g * 4 + r;
        if (t < sp.count) a.out[static_cast<size_t>(sp.first + t) * (static_cast<size_t>(a.H) * a.dv) + static_cast<size_t>(h) * a.dv + col] = result[r];
      }
    }
    src = next;
  }
#pragma unroll
  for (int n = 0; n < NW; ++n) {
    const int d = (wave * NW + n) * 16 + g * 4;
    if (col_ok && d < a.dk) *reinterpret_cast<floatx4*>(S + static_cast<size_t>(col) * a.dk + d) = s[n];
  }
}

// The walk for the state alone, which keeps the state in front of each piece for piece_outputs_kernel: a wave per head and block of 16
// channels x 16 columns, and no barriers, as no wave needs another's part.  What a piece adds does not need the state, so that its
// products run ahead of the chain, which is one multiply-add a piece.
template <int NT>
__global__ __launch_bounds__(256, 2) void linear_scan_kernel(Args a) {
  constexpr int AHEAD = 3;   // pieces whose operands are asked for
  const Span sp = span_of(a.seq_meta, a.row0, a.row1, blockIdx.z);
  if (sp.count <= 0) return;
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid % kWave;
  const int job = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(tid / kWave), n = job % NT, cbk = job / NT;
  const int c = lane % 16, g = lane / 16, col = cbk * 16 + c, d = n * 16 + g * 4, count = (sp.count + kTokens - 1) / kTokens;
  const bool ok = col < a.dv && d < a.dk;
  const Layout lay = layout(NT, (a.dv + 15) / 16, true);
  float* piece = a.pieces + (static_cast<size_t>(sp.piece0) * a.H + h) * lay.words;
  const size_t step = static_cast<size_t>(a.H) * lay.words;
  float* S = a.state + static_cast<size_t>(sp.slot) * a.state_stride + static_cast<size_t>(h) * a.dk * a.dv + static_cast<size_t>(col) * a.dk + d;
  floatx4 s{0.f, 0.f, 0.f, 0.f};
  if (ok) s = *reinterpret_cast<const floatx4*>(S);
  floatx4 kt[AHEAD][kBlocks], v[AHEAD][kBlocks], all[AHEAD];
  auto fetch = [&](int i, int of) __attribute__((always_inline)) {   // (behind the last piece: that one again, for nothing)
    const float* from = piece + (of < count ? of : count - 1) * step;
    all[i] = *reinterpret_cast<const floatx4*>(from + lay.all + d);
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
      kt[i][b] = *reinterpret_cast<const floatx4*>(from + lay.kt + (n * kBlocks + b) * kBlock + lane * 4);
      v[i][b] = *reinterpret_cast<const floatx4*>(from + lay.v + (cbk * kBlocks + b) * kBlock + lane * 4);
    }
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) fetch(i, i);
  for (int at = 0; at < count; at += AHEAD) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (at + i >= count) break;   // (uniform)
      floatx4 more[kBlocks];
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) more[b] = mul4(kt[i][b], v[i][b], floatx4{0.f, 0.f, 0.f, 0.f});
      const floatx4 added = ((more[0] + more[1]) + more[2]) + more[3], decays = all[i];
      *reinterpret_cast<floatx4*>(piece + (at + i) * step + lay.states + (cbk * NT + n) * kBlock + lane * 4) = s;
      fetch(i, at + i + AHEAD);
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = fmaf(s[r], decays[r], added[r]);
    }
  }
  if (ok) *reinterpret_cast<floatx4*>(S) = s;
}

}  // namespace linear
}  // namespace sa

using namespace sa;

static int64_t linear_piece_bytes(int H, int dk, int dv, bool keep = false) {
  return static_cast<int64_t>(H) * linear::layout(dk <= 64 ? 4 : 8, (dv + 15) / 16, keep).words * static_cast<int64_t>(sizeof(float));
}

extern "C" int sa_linear_chunks_takes(int H, int dk, int dv, int q_at, int k_at, int64_t proj_stride, int64_t gates_stride,
                                      int64_t state_stride, int num_seqs, int64_t workspace_bytes) {
  return H > 0 && H <= 65535 && dk > 0 && dk <= 128 && dk % 4 == 0 && dv > 0 && dv <= 16 * 65535 && q_at % 4 == 0 &&
         k_at % 4 == 0 && proj_stride % 4 == 0 && gates_stride % 4 == 0 && state_stride % 4 == 0 && num_seqs > 0 &&
         num_seqs <= 65535 && (num_seqs + 1) * linear_piece_bytes(H, dk, dv) <= workspace_bytes;
}

extern "C" int sa_linear_chunks(const void* proj, int64_t proj_stride, int q_at, int k_at, int v_at, float q_mult,
                                const float* gates, int64_t gates_stride, const void* gate_bias, int bias_dtype, float tau,
                                const void* bonus, int bonus_dtype, int H, int dk, int dv, float* state, int64_t state_stride,
                                const int* seq_meta, int num_seqs, int first_row, int rows, int max_q_len, float* out,
                                void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  if (num_seqs == 0 || rows == 0) return 0;
  SA_REQUIRE(num_seqs > 0 && H > 0 && dk > 0 && dv > 0 && first_row >= 0 && rows > 0 && max_q_len > 0 && tau >= 0.f,
             "linear_chunks: bad sizes S=%d H=%d dk=%d dv=%d", num_seqs, H, dk, dv);
  SA_REQUIRE(proj != nullptr && gates != nullptr && state != nullptr && seq_meta != nullptr && out != nullptr && workspace != nullptr &&
                 reinterpret_cast<uintptr_t>(proj) % 8 == 0 && reinterpret_cast<uintptr_t>(gates) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(state) % 16 == 0 && reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
             "linear_chunks: a null or unaligned pointer");
  SA_REQUIRE(q_at >= 0 && k_at >= 0 && v_at >= 0 && proj_stride >= q_at + static_cast<int64_t>(H) * dk &&
                 proj_stride >= k_at + static_cast<int64_t>(H) * dk && proj_stride >= v_at + static_cast<int64_t>(H) * dv &&
                 gates_stride >= static_cast<int64_t>(H) * dk && state_stride >= static_cast<int64_t>(H) * dk * dv,
             "linear_chunks: rows of the projection, the gates or the state are too short");
  SA_REQUIRE((gate_bias == nullptr || bias_dtype == kF32 || bias_dtype == kBF16) &&
                 (bonus == nullptr || bonus_dtype == kF32 || bonus_dtype == kBF16) && (bonus == nullptr || tau == 0.f),
             "linear_chunks: unknown dtype, or a bonus with tau");
  SA_REQUIRE(sa_linear_chunks_takes(H, dk, dv, q_at, k_at, proj_stride, gates_stride, state_stride, num_seqs, workspace_bytes),
             "linear_chunks: does not take keys of %d and values of %d, %d requests", dk, dv, num_seqs);
  linear::Args a;
  a.proj = static_cast<const bf16*>(proj), a.gates = gates, a.gate_bias = gate_bias, a.bonus = bonus, a.state = state, a.out = out;
  a.pieces = static_cast<float*>(workspace), a.seq_meta = seq_meta, a.proj_stride = proj_stride, a.gates_stride = gates_stride;
  a.state_stride = state_stride, a.q_mult = q_mult, a.inv_tau = tau > 0.f ? 1.f / tau : 0.f, a.q_at = q_at, a.k_at = k_at;
  a.v_at = v_at, a.H = H, a.dk = dk, a.dv = dv, a.bias_dtype = bias_dtype, a.bonus_dtype = bonus_dtype;
  a.keep = chunks::keeps_states(max_q_len, static_cast<int64_t>(H) * ((dv + 15) / 16) * num_seqs) &&
           rows / chunks::kTokens + num_seqs < workspace_bytes / linear_piece_bytes(H, dk, dv, true);
  // as many rows at a time as the workspace has room for: R rows are at most R / 64 + num_seqs pieces
  const int64_t room = (workspace_bytes / linear_piece_bytes(H, dk, dv, a.keep) - num_seqs) * chunks::kTokens;
  const int span = static_cast<int>(room < rows ? room : rows);
  for (int r = 0; r < rows; r += span) {
    a.row0 = first_row + r;
    a.row1 = first_row + (r + span < rows ? r + span : rows);
    const int longest = a.row1 - a.row0 < max_q_len ? a.row1 - a.row0 : max_q_len;
    const dim3 pieces(H, (longest + chunks::kTokens - 1) / chunks::kTokens, num_seqs), walk(H, (dv + 15) / 16, num_seqs);
#define SA_LINEAR(NT)                                                                              \
  do {                                                                                             \
    if (bonus != nullptr) linear::linear_pieces_kernel<NT, true><<<pieces, 256, 0, stream>>>(a);   \
    else linear::linear_pieces_kernel<NT, false><<<pieces, 256, 0, stream>>>(a);                   \
    if (a.keep) {                                                                                  \
      const linear::Layout lay = linear::layout(NT, (dv + 15) / 16, true);                         \
      const chunks::OutputsAt at{lay.q, lay.p, lay.v, lay.states, 0, lay.words};                   \
      linear::linear_scan_kernel<NT><<<dim3(H, (dv + 15) / 16 * (NT / 4), num_seqs), 256, 0, stream>>>(a); \
      chunks::piece_outputs_kernel<NT, false><<<pieces, 256, 0, stream>>>(a.pieces, at, seq_meta, a.row0, a.row1, H, dv, out); \
    } else {                                                                                       \
      linear::linear_walk_kernel<NT><<<walk, 256, 0, stream>>>(a);                                 \
    }                                                                                              \
  } while (0)
    if (dk <= 64) SA_LINEAR(4);
    else SA_LINEAR(8);
#undef SA_LINEAR
  }
  return check_launch("linear_chunks");
}
