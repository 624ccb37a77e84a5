// The gated delta rule of delta_rule.hip for portions of prompts, on the matrix cores: 64 tokens (a piece) at a time.  With
// L_i the sum of the decays' logarithms up to token i of a piece and S the state in front of it, the rule's
//
//   S_i = g_i S_(i-1) + k_i u_i^T,   u_i = beta_i (v_i - g_i S_(i-1)^T k_i),   o_i = S_i^T q_i
//
// is a system with a unit lower triangular matrix, A_ij = beta_i exp(L_i - L_j) (k_i . k_j) for j < i:
//
//   (I + A) U = diag(beta) V - diag(beta_i exp(L_i)) K S     =>   U = U0 - W S,
//   (I + A) [W | U0] = [diag(beta_i exp(L_i)) K | diag(beta) V]
//   o_i = exp(L_i) S^T q_i + sum_(j <= i) P_ij u_j,          P_ij = exp(L_i - L_j) (q_i . k_j)
//   S  <- exp(L_64) S + sum_j exp(L_64 - L_j) k_j u_j^T
//
// (the form that is known from chunked linear recurrences as the WY representation of a product of rank-one updates).
//
//   delta_pieces_kernel   everything that does not need the state, a workgroup per piece and head: the products of keys and
//                         queries, the solution W, U0 by blocks of 16 rows (the blocks on the diagonal inverted by
//                         substitution, the others by products), and all operands of the second kernel, scaled, in the
//                         order in which its matrix instructions take them, into the workspace
//   delta_state_kernel    the walk through the pieces, a workgroup of four waves per head and 16 value columns; or, for long
//                         requests of few heads (keeps_states), delta_walk_kernel for the state alone and piece_outputs_kernel
//
// Everything is 32-bit: products are v_mfma_f32_16x16x4_f32, sums of logarithms 64-bit.  A 16 x 16 result holds rows
// 4 g + r (g = lane / 16) and column lane % 16; an operand of step r holds k = 4 g + r, so that a result is the next
// product's right operand as it lies in registers (U0 - W S, then P U and K^T U), and left operands are 16 bytes a lane.
// In delta_state_kernel wave w owns tokens 16 w .. 16 w + 15 of a piece for W S, Q S and P U, and a quarter of the key
// channels of the state, kept in registers and, for the other waves, in LDS.  The next piece's operands are asked for while
// this one is worked through.  Bound by the matrix instructions that a wave issues one after the other (about 110 of 32
// clocks a piece) and two barriers a piece, on as many CUs as there are heads times blocks of 16 columns.
//
// Long chains of matrix instructions round at the size of the sum with every product, so sums run in several short chains, the
// state's increment and the entries on the diagonal by themselves.  The error against 64 bits is then that of delta_rule.hip
// (rates and steps as in models of the kind, 64 to 2,048 tokens: results 0.57 to 1.05 times, the state 0.4 to 0.87 times; with
// decays drawn evenly from 0 to 1, half-lives of a token, 1.2 and 1.2 to 1.4 times, and no less with exponentials in 64 bits);
// with one or two chains each results were off by up to twice as much.
//
// Measured at 2,048 tokens of 16 heads over 8, sizes 128: 121 us (traced, 50 for the pieces, 60 for the walk of the state, 29 for the
// outputs; 137 with delta_state_kernel's 106 instead), where delta_rule.hip takes 589 token by token.
#include "api.h"
#include "chunks.h"

namespace sa {
namespace delta {

using namespace chunks;

// A piece's operands in the workspace (floats), for NT blocks of 16 key channels and CB blocks of 16 value columns.
struct Layout {
  int w, q, kt, p, u0, decay, own, states, words;   // states: in front of the pieces, where they are kept
};
__host__ __device__ constexpr Layout layout(int nt, int cb, bool keep) {
  Layout l{};
  l.w = 0;                             // [token block][channel block]
  l.q = l.w + kBlocks * nt * kBlock;   // likewise
  l.kt = l.q + kBlocks * nt * kBlock;  // [channel block][token block]
  l.p = l.kt + kBlocks * nt * kBlock;  // [token block][token block], without the diagonal
  l.u0 = l.p + kBlocks * kBlocks * kBlock;   // [column block][token block]; where states are kept, then U
  l.decay = l.u0 + cb * kBlocks * kBlock;    // exp(L_64)
  l.own = l.decay + 64;                      // the diagonal of P
  l.states = l.own + kTokens;                // [column block][channel block]
  l.words = l.states + (keep ? cb * nt * kBlock : 0);
  return l;
}

struct Args {
  const float* qkv;     // [T, C]: q heads, k heads (G of them each), values
  const float* gates;   // [T, 2 H]: beta, decay
  float* state;         // per slot and head [dv][dk]
  float* out;           // [T, H * dv]
  float* pieces;
  const int* seq_meta;
  int64_t state_stride;
  int C, G, H, dk, dv, row0, row1;   // the rows of the step that this launch is about
  bool keep;            // the states in front of the pieces
};

// exp(x) for x <= 0; what 32 bits do not hold of x goes in as a factor (a rounding of x alone would be |x| of them of exp(x)).
__device__ __forceinline__ float decay_between(double x) {
  const float hi = static_cast<float>(x), e = expf(hi);
  return fmaf(e, static_cast<float>(x - static_cast<double>(hi)), e);
}

template <int NT>
__global__ __launch_bounds__(256) void delta_pieces_kernel(Args a) {
  constexpr int ROW = NT * 16 + 4, AROW = kTokens + 4, QUADS = NT * 4;
  __shared__ __align__(16) float k_s[kTokens * ROW];
  __shared__ __align__(16) float q_s[kTokens * ROW];   // rows of q; then A, then its diagonal blocks' inverses beside it
  __shared__ double cum_s[kTokens];
  __shared__ float beta_s[kTokens], in_s[kTokens], out_s[kTokens];   // beta, exp(L_i), exp(L_64 - L_i)
  static_assert(kTokens * ROW >= kTokens * AROW || NT < 4, "A lies where q lay");
  const Span sp = span_of(a.seq_meta, a.row0, a.row1, blockIdx.z);
  const int t0 = blockIdx.y * kTokens;
  if (t0 >= sp.count) return;   // (uniform)
  const int left = sp.count - t0 < kTokens ? sp.count - t0 : kTokens;
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), c = lane % 16, g = lane / 16;
  const int qk = h / (a.H / a.G), row0 = sp.first + t0;
  const Layout lay = layout(NT, (a.dv + 15) / 16, a.keep);
  float* dst = a.pieces + (static_cast<size_t>(sp.piece0 + blockIdx.y) * a.H + h) * lay.words;

  // rows of q and k (tokens behind the last, channels behind the last: zeros)
#pragma unroll
  for (int i = 0; i < kTokens * QUADS / 256; ++i) {
    const int idx = tid + i * 256, j = idx / QUADS, d = idx % QUADS * 4;
    floatx4 kv{0.f, 0.f, 0.f, 0.f}, qv{0.f, 0.f, 0.f, 0.f};
    if (j < left && d < a.dk) {
      const float* row = a.qkv + static_cast<size_t>(row0 + j) * a.C;
      qv = *reinterpret_cast<const floatx4*>(row + qk * a.dk + d);
      kv = *reinterpret_cast<const floatx4*>(row + (a.G + qk) * a.dk + d);
    }
    *reinterpret_cast<floatx4*>(&k_s[j * ROW + d]) = kv;
    *reinterpret_cast<floatx4*>(&q_s[j * ROW + d]) = qv;
  }
  if (wave == 0) {
    const bool live = lane < left;
    const float* gr = a.gates + static_cast<size_t>(row0 + (live ? lane : 0)) * 2 * a.H + h;
    const float beta = live ? gr[0] : 0.f, decay = live ? gr[a.H] : 1.f;
    // (a decay of zero: a logarithm whose exponential is zero, so that differences stay defined)
    double cum = decay > 0.f ? log(static_cast<double>(decay)) : decay == 0.f ? -1e4 : static_cast<double>(decay) * NAN;
#pragma unroll
    for (int by = 1; by < kWave; by *= 2) {
      const double up = __shfl_up(cum, by, kWave);
      if (lane >= by) cum += up;
    }
    const double end = __shfl(cum, kWave - 1, kWave);
    cum_s[lane] = cum;
    beta_s[lane] = beta;
    in_s[lane] = decay_between(cum);
    out_s[lane] = decay_between(end - cum);
    if (lane == 0) dst[lay.decay] = decay_between(end);
  }
  __syncthreads();

  // products of rows: P as [key token 4 g + r, query token c], which is the left operand's order, for key blocks b <= wave;
  // k . k as [token 4 g + r, earlier token c], to become A
  floatx4 kk[kBlocks];
  const double cum_c = cum_s[wave * 16 + c];
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
    kk[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (b <= wave) {   // (uniform over the wave)
      floatx4 qk_b[NT], kk_b[NT];   // (a chain of products for each 16 channels)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const floatx4 kb = *reinterpret_cast<const floatx4*>(&k_s[(b * 16 + c) * ROW + n * 16 + g * 4]);
        const floatx4 kw = *reinterpret_cast<const floatx4*>(&k_s[(wave * 16 + c) * ROW + n * 16 + g * 4]);
        const floatx4 qw = *reinterpret_cast<const floatx4*>(&q_s[(wave * 16 + c) * ROW + n * 16 + g * 4]);
        qk_b[n] = mul4(kb, qw, kk[b]);
        kk_b[n] = mul4(kw, kb, kk[b]);
      }
      const floatx4 qk_all = sum_of(qk_b);
      kk[b] = sum_of(kk_b);
      floatx4 p;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = b * 16 + g * 4 + r, i = wave * 16 + c;
        p[r] = j < i ? qk_all[r] * decay_between(cum_c - cum_s[j]) : 0.f;
        if (j == i) dst[lay.own + i] = qk_all[r];
      }
      *reinterpret_cast<floatx4*>(dst + lay.p + (wave * kBlocks + b) * kBlock + lane * 4) = p;
    }
  }
  // the queries times exp(L_i), and the keys times exp(L_64 - L_j), turned
  {
    const float e = in_s[wave * 16 + c];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const floatx4 q = *reinterpret_cast<const floatx4*>(&q_s[(wave * 16 + c) * ROW + n * 16 + g * 4]);
      *reinterpret_cast<floatx4*>(dst + lay.q + (wave * NT + n) * kBlock + lane * 4) = floatx4{q[0] * e, q[1] * e, q[2] * e, q[3] * e};
      floatx4 kt;
#pragma unroll
      for (int r = 0; r < 4; ++r) kt[r] = k_s[(wave * 16 + g * 4 + r) * ROW + n * 16 + c] * out_s[wave * 16 + g * 4 + r];
      *reinterpret_cast<floatx4*>(dst + lay.kt + (n * kBlocks + wave) * kBlock + lane * 4) = kt;
    }
  }
  __syncthreads();   // (q has been read)
  float* a_s = q_s;
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
    if (b <= wave) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = wave * 16 + g * 4 + r, j = b * 16 + c;
        a_s[i * AROW + j] = j < i ? kk[b][r] * beta_s[i] * decay_between(cum_s[i] - cum_s[j]) : 0.f;
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // the inverse of the wave's diagonal block: lane c solves for column c (the four groups of lanes alike)
  {
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s[4] = {i == c ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j4 = 0; j4 < (i + 3) / 4; ++j4) {
        const floatx4 row = *reinterpret_cast<const floatx4*>(&a_s[(wave * 16 + i) * AROW + wave * 16 + j4 * 4]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j4 * 4 + e < i) s[e] = fmaf(-row[e], x[j4 * 4 + e], s[e]);
      }
      x[i] = (s[0] + s[1]) + (s[2] + s[3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // into the block's own place (its entries have been read), without the ones on the diagonal: a sum of 16 products that
    // holds the large one rounds at its size 16 times
    if (g == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) a_s[(wave * 16 + i) * AROW + wave * 16 + c] = i == c ? 0.f : x[i];
    }
  }
  __syncthreads();
  // W and U0, 16 columns at a time: channels first, then value columns
  const int cb = (a.dv + 15) / 16;
  for (int n = wave; n < NT + cb; n += 4) {
    floatx4 x[kBlocks];
    const int col = (n - NT) * 16 + c;
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
      floatx4 acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = b * 16 + g * 4 + r;
        if (n < NT) acc[r] = k_s[i * ROW + n * 16 + c] * (beta_s[i] * in_s[i]);
        else acc[r] = (i < left && col < a.dv) ? a.qkv[static_cast<size_t>(row0 + i) * a.C + 2 * a.G * a.dk + h * a.dv + col] * beta_s[i] : 0.f;
      }
      floatx4 less[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int e = 0; e < b; ++e)
        less[e % 2] = mul4(*reinterpret_cast<const floatx4*>(&a_s[(b * 16 + c) * AROW + e * 16 + g * 4]), x[e], less[e % 2]);
      acc -= less[0] + less[1];
      const floatx4 inv = *reinterpret_cast<const floatx4*>(&a_s[(b * 16 + c) * AROW + b * 16 + g * 4]);
      x[b] = acc + lower_mul4<false>(inv, acc, floatx4{0.f, 0.f, 0.f, 0.f}, lane);
    }
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
      if (n < NT) {   // as a left operand: [token c][channels 4 g ..]; this lane has channel c of tokens 4 g + r
        float* to = dst + lay.w + (b * NT + n) * kBlock + (c / 4) * 64 + c % 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) to[(g * 4 + r) * 4] = x[b][r];
      } else {
        *reinterpret_cast<floatx4*>(dst + lay.u0 + ((n - NT) * kBlocks + b) * kBlock + lane * 4) = x[b];
      }
    }
  }
}

template <int NT>
__global__ __launch_bounds__(256) void delta_state_kernel(Args a) {
  constexpr int NW = NT / 4;   // blocks of key channels whose state a wave holds
  __shared__ __align__(16) floatx4 s_s[2][NT * kWave];
  __shared__ __align__(16) floatx4 u_s[kBlocks * kWave];
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
  floatx4 w[NT], q[NT], kt[NW][kBlocks], p[kBlocks], u0, own;   // (p: blocks in front of the wave's own, and that)
  float all;
  auto fetch_state = [&](const float* from) __attribute__((always_inline)) {   // what U and the state behind the piece need
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n] = *reinterpret_cast<const floatx4*>(from + lay.w + (wave * NT + n) * kBlock + lane * 4);
    u0 = *reinterpret_cast<const floatx4*>(from + lay.u0 + (blockIdx.y * kBlocks + wave) * kBlock + lane * 4);
  };
  auto fetch_rest = [&](const float* from) __attribute__((always_inline)) {
    all = from[lay.decay];
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
      for (int b = 0; b < kBlocks; ++b)
        kt[n][b] = *reinterpret_cast<const floatx4*>(from + lay.kt + ((wave * NW + n) * kBlocks + b) * kBlock + lane * 4);
#pragma unroll
    for (int n = 0; n < NT; ++n) q[n] = *reinterpret_cast<const floatx4*>(from + lay.q + (wave * NT + n) * kBlock + lane * 4);
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {   // (the last: the wave's own; others behind it: that again, not used)
      const int at = b < wave ? b : wave;
      p[b] = *reinterpret_cast<const floatx4*>(from + lay.p + (wave * kBlocks + at) * kBlock + lane * 4);
    }
    own = *reinterpret_cast<const floatx4*>(from + lay.own + wave * 16 + g * 4);
  };
  fetch_state(src);
  fetch_rest(src);
  int now = 0;
  for (int t0 = 0; t0 < sp.count; t0 += kTokens, now ^= 1) {
    // (behind the last piece: that one again, for nothing)
    const float* next = t0 + kTokens < sp.count ? src + step : src;
    __syncthreads();   // the state in front of the piece is there
    floatx4 st[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) st[n] = s_s[now][n * kWave + lane];
    // (sums in four chains, and the state's increment by itself: 64 products added to the state one by one would round it
    // 64 times)
    floatx4 x[4], o[4], o2[kBlocks], more[2][NW];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) o2[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < NT; n += 4)
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = mul4(w[n + i], st[n + i], x[i]);
    const floatx4 u = u0 - sum_of(x);
    u_s[wave * kWave + lane] = u;
    fetch_state(next);
#pragma unroll
    for (int n = 0; n < NT; n += 4)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = mul4(q[n + i], st[n + i], o[i]);
    __syncthreads();
    floatx4 ub[kBlocks];
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) ub[b] = u_s[b * kWave + lane];
#pragma unroll
    for (int n = 0; n < NW; ++n) more[0][n] = more[1][n] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < kBlocks; ++b)
#pragma unroll
      for (int n = 0; n < NW; ++n) more[b % 2][n] = mul4(kt[n][b], ub[b], more[b % 2][n]);
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[n][r] = fmaf(s[n][r], all, more[0][n][r] + more[1][n][r]);
#pragma unroll
    for (int n = 0; n < NW; ++n) s_s[now ^ 1][(wave * NW + n) * kWave + lane] = s[n];
#pragma unroll
    for (int b = 0; b < kBlocks - 1; ++b)
      if (b < wave) o2[b] = mul4(p[b], ub[b], o2[b]);   // (uniform over the wave)
    o2[kBlocks - 1] = lower_mul4<false>(p[kBlocks - 1], u, o2[kBlocks - 1], lane);
    floatx4 result = sum_of(o) + sum_of(o2);
#pragma unroll
    for (int r = 0; r < 4; ++r) result[r] = fmaf(own[r], u[r], result[r]);
    if (col_ok) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + wave * 16 + g * 4 + r;
        if (t < sp.count) a.out[static_cast<size_t>(sp.first + t) * (static_cast<size_t>(a.H) * a.dv) + static_cast<size_t>(h) * a.dv + col] = result[r];
      }
    }
    fetch_rest(next);
    src = next;
  }
#pragma unroll
  for (int n = 0; n < NW; ++n) {
    const int d = (wave * NW + n) * 16 + g * 4;
    if (col_ok && d < a.dk) *reinterpret_cast<floatx4*>(S + static_cast<size_t>(col) * a.dk + d) = s[n];
  }
}

// The walk for the state alone: the same sums, and U and the state in front of each piece are kept for piece_outputs_kernel.  Of 110
// matrix instructions a wave issues 64 a piece; the next piece's operands are asked for, and what is kept is written, among the
// products of the state's increment.  (Operands of two pieces ahead, in twice the registers, were slower: 66 us instead of 60.)
template <int NT>
__global__ __launch_bounds__(256) void delta_walk_kernel(Args a) {
  constexpr int NW = NT / 4;   // blocks of key channels whose state a wave holds
  __shared__ __align__(16) floatx4 s_s[2][NT * kWave];
  __shared__ __align__(16) floatx4 u_s[kBlocks * kWave];
  const Span sp = span_of(a.seq_meta, a.row0, a.row1, blockIdx.z);
  if (sp.count <= 0) return;
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), c = lane % 16, g = lane / 16;
  const int col = blockIdx.y * 16 + c, count = (sp.count + kTokens - 1) / kTokens;
  const bool col_ok = col < a.dv;
  const Layout lay = layout(NT, (a.dv + 15) / 16, true);
  float* first = a.pieces + (static_cast<size_t>(sp.piece0) * a.H + h) * lay.words;
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
  floatx4 w[NT], kt[NW][kBlocks], u0;
  float all;
  // a piece's operands, asked for a piece ahead
  auto fetch_w = [&](const float* from, int n) __attribute__((always_inline)) {
    w[n] = *reinterpret_cast<const floatx4*>(from + lay.w + (wave * NT + n) * kBlock + lane * 4);
  };
  auto fetch_kt = [&](const float* from, int n, int b) __attribute__((always_inline)) {
    kt[n][b] = *reinterpret_cast<const floatx4*>(from + lay.kt + ((wave * NW + n) * kBlocks + b) * kBlock + lane * 4);
  };
  auto fetch_rest = [&](const float* from) __attribute__((always_inline)) {
    u0 = *reinterpret_cast<const floatx4*>(from + lay.u0 + (blockIdx.y * kBlocks + wave) * kBlock + lane * 4);
    all = from[lay.decay];
  };
#pragma unroll
  for (int n = 0; n < NT; ++n) fetch_w(first, n);
#pragma unroll
  for (int n = 0; n < NW; ++n)
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) fetch_kt(first, n, b);
  fetch_rest(first);
  for (int at = 0; at < count; at += 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (at + i >= count) break;   // (uniform)
      float* piece = first + (at + i) * step;
      // (behind the last piece: that one again, for nothing; its U0 may have become U)
      const float* from = at + i + 1 < count ? piece + step : piece;
      __syncthreads();   // the state in front of the piece is there
      floatx4 st[NT], x[4], more[2][NW];
#pragma unroll
      for (int n = 0; n < NT; ++n) st[n] = s_s[i][n * kWave + lane];
      __builtin_amdgcn_sched_barrier(0);   // (all reads are under way before the first product)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < NT; n += 4)
#pragma unroll
        for (int r = 0; r < 4; ++r)   // (the four chains in turn)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            x[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[n + e][r], st[n + e][r], x[e], 0, 0, 0);
      const floatx4 u = u0 - sum_of(x);
      u_s[wave * kWave + lane] = u;
      __syncthreads();
      floatx4 ub[kBlocks];
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) ub[b] = u_s[b * kWave + lane];
#pragma unroll
      for (int n = 0; n < NW; ++n) more[0][n] = more[1][n] = floatx4{0.f, 0.f, 0.f, 0.f};
      const float decay = all;
      // memory is asked for among these products, one access after every few: nothing but LDS stands between the others' u and x
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < kBlocks; b += 2) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int n = 0; n < NW; ++n)
              more[e][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[n][b + e][r], ub[b + e][r], more[e][n], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (b / 2 * 4 + r < NT) fetch_w(from, b / 2 * 4 + r);
          if (b == 0 && r < NW)
            *reinterpret_cast<floatx4*>(piece + lay.states + (blockIdx.y * NT + wave * NW + r) * kBlock + lane * 4) = s[r];
          if (b == 0 && r == 3) *reinterpret_cast<floatx4*>(piece + lay.u0 + (blockIdx.y * kBlocks + wave) * kBlock + lane * 4) = u;
          if (b == 2 && r < NW) {
            fetch_kt(from, r, 0);
            fetch_kt(from, r, 1);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int n = 0; n < NW; ++n) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s[n][r] = fmaf(s[n][r], decay, more[0][n][r] + more[1][n][r]);
        s_s[i ^ 1][(wave * NW + n) * kWave + lane] = s[n];
      }
#pragma unroll
      for (int n = 0; n < NW; ++n) {
        fetch_kt(from, n, 2);
        fetch_kt(from, n, 3);
      }
      fetch_rest(from);
    }
  }
#pragma unroll
  for (int n = 0; n < NW; ++n) {
    const int d = (wave * NW + n) * 16 + g * 4;
    if (col_ok && d < a.dk) *reinterpret_cast<floatx4*>(S + static_cast<size_t>(col) * a.dk + d) = s[n];
  }
}

}  // namespace delta
}  // namespace sa

using namespace sa;

static int64_t delta_piece_bytes(int H, int dk, int dv, bool keep = false) {
  return static_cast<int64_t>(H) * delta::layout(dk <= 64 ? 4 : 8, (dv + 15) / 16, keep).words * static_cast<int64_t>(sizeof(float));
}

extern "C" int sa_delta_chunks_takes(int C, int G, int H, int dk, int dv, int64_t state_stride, int num_seqs, int64_t workspace_bytes) {
  return G > 0 && H > 0 && H % G == 0 && H <= 65535 && dk > 0 && dk <= 128 && dk % 4 == 0 && dv > 0 && dv <= 16 * 65535 &&
         C % 4 == 0 && state_stride % 4 == 0 && num_seqs > 0 && num_seqs <= 65535 &&
         (num_seqs + 1) * delta_piece_bytes(H, dk, dv) <= workspace_bytes;
}

extern "C" int sa_delta_chunks(const float* qkv, int C, int G, int dk, int dv, const float* gates, int H, float* state,
                               int64_t state_stride, const int* seq_meta, int num_seqs, int first_row, int rows, int max_q_len,
                               float* out, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  if (num_seqs == 0 || rows == 0) return 0;
  SA_REQUIRE(num_seqs > 0 && G > 0 && H > 0 && H % G == 0 && dk > 0 && dv > 0 && C >= 2 * G * dk + H * dv && first_row >= 0 &&
                 rows > 0 && max_q_len > 0,
             "delta_chunks: bad sizes S=%d C=%d G=%d H=%d dk=%d dv=%d", num_seqs, C, G, H, dk, dv);
  SA_REQUIRE(qkv != nullptr && gates != nullptr && state != nullptr && seq_meta != nullptr && out != nullptr && workspace != nullptr &&
                 reinterpret_cast<uintptr_t>(qkv) % 16 == 0 && reinterpret_cast<uintptr_t>(state) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
             "delta_chunks: a null or unaligned pointer");
  SA_REQUIRE(state_stride >= static_cast<int64_t>(H) * dk * dv, "delta_chunks: the state rows are too short");
  SA_REQUIRE(sa_delta_chunks_takes(C, G, H, dk, dv, state_stride, num_seqs, workspace_bytes),
             "delta_chunks: does not take keys of %d and values of %d, %d requests", dk, dv, num_seqs);
  delta::Args a;
  a.qkv = qkv, a.gates = gates, a.state = state, a.out = out, a.pieces = static_cast<float*>(workspace), a.seq_meta = seq_meta;
  a.state_stride = state_stride, a.C = C, a.G = G, a.H = H, a.dk = dk, a.dv = dv;
  a.keep = chunks::keeps_states(max_q_len, static_cast<int64_t>(H) * ((dv + 15) / 16) * num_seqs) &&
           rows / chunks::kTokens + num_seqs < workspace_bytes / delta_piece_bytes(H, dk, dv, true);
  // as many rows at a time as the workspace has room for: R rows are at most R / 64 + num_seqs pieces
  const int64_t room = (workspace_bytes / delta_piece_bytes(H, dk, dv, a.keep) - num_seqs) * chunks::kTokens;
  const int span = static_cast<int>(room < rows ? room : rows);
  for (int r = 0; r < rows; r += span) {
    a.row0 = first_row + r;
    a.row1 = first_row + (r + span < rows ? r + span : rows);
    const int longest = a.row1 - a.row0 < max_q_len ? a.row1 - a.row0 : max_q_len;
    const dim3 pieces(H, (longest + chunks::kTokens - 1) / chunks::kTokens, num_seqs), walk(H, (dv + 15) / 16, num_seqs);
#define SA_DELTA(NT)                                                                               \
  do {                                                                                             \
    delta::delta_pieces_kernel<NT><<<pieces, 256, 0, stream>>>(a);                                 \
    if (a.keep) {                                                                                  \
      const delta::Layout lay = delta::layout(NT, (dv + 15) / 16, true);                           \
      const chunks::OutputsAt at{lay.q, lay.p, lay.u0, lay.states, lay.own, lay.words};            \
      delta::delta_walk_kernel<NT><<<walk, 256, 0, stream>>>(a);                            \
      chunks::piece_outputs_kernel<NT, true><<<pieces, 256, 0, stream>>>(a.pieces, at, seq_meta, a.row0, a.row1, H, dv, out); \
    } else {                                                                                       \
      delta::delta_state_kernel<NT><<<walk, 256, 0, stream>>>(a);                           \
    }                                                                                              \
  } while (0)
    if (dk <= 64) SA_DELTA(4);
    else SA_DELTA(8);
#undef SA_DELTA
  }
  return check_launch("delta_chunks");
}
