// Row-wise kernels of blocks that norm a part's output instead of its input, and of mixers with gates:
//   residual += mult * norm(y)  and the residual handed on in the activation type (no norm in front of the next part);
//   heads normed one by one and multiplied by a gate, sigmoid(g) or silu(g);
//   an activation applied to a product in place;
//   queries and keys rotated on their first dimensions only, then divided by their root mean square, values mixed
//   with those of an earlier layer, keys and values written into pages whose value size differs from the key size.
// Statistics, angles and sums are 32-bit whatever the activation type is; square roots and divisions are the
// correctly rounded ones (no reciprocal-square-root instruction).
#include "api.h"
#include "common.h"
#include "eights.h"

namespace sa {

// Eight neighbouring entries of a row in two registers of 16 bytes (32-bit) or one (bfloat16); a thread's pieces of a row are
// 8 (p 256 + thread) .. + 7.  Rows whose width and strides are multiples of 8 and whose pointers are aligned are read so: every
// load is unconditional (a piece behind the row's end stands for the row's last one), so that a row's loads are all under way
// together.  Layer norm of eight rows of 2,048 with the sum: 10.3 us with an entry at a time behind a test of the row's end, 4.6
// in pieces (launch and two waits for memory); of 2,047 rows 16.5 and 11.2 us (50 MB: 4.5 TB/s), the sum of normed rows 13.0 and
// 10.8.
static bool rows_in_eights(int D, int64_t y_stride, const void* a, const void* b, const void* c, const void* d, const void* e) {
  return D % 8 == 0 && y_stride % 8 == 0 &&
         ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(d) |
           reinterpret_cast<uintptr_t>(e)) & 15u) == 0;
}

// ------------------------------------------------------------------ residual += mult * norm(y); out = residual
// y null: nothing is added (the residual is only handed on in out's type).  out null: nothing is handed on.
__global__ __launch_bounds__(256) void residual_add_norm_kernel(
    const void* __restrict__ y, int y_dtype, int64_t y_stride, const void* __restrict__ w, int w_dtype, float eps,
    float plus_one, float mult, float* __restrict__ residual, void* __restrict__ out, int out_dtype, int D) {
  __shared__ float scratch[16];
  const size_t yb = static_cast<size_t>(blockIdx.x) * y_stride, rb = static_cast<size_t>(blockIdx.x) * D;
  if (y == nullptr) {
    for (int d = threadIdx.x; d < D; d += blockDim.x) store_f(out, out_dtype, rb + d, residual[rb + d]);
    return;
  }
  float r = 1.f;
  if (w != nullptr) {
    float ss = 0.f;
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
      const float v = load_f(y, y_dtype, yb + d);
      ss = fmaf(v, v, ss);
    }
    ss = block_sum(ss, scratch);
    r = 1.f / sqrtf(ss / static_cast<float>(D) + eps);
  }
  for (int d = threadIdx.x; d < D; d += blockDim.x) {
    float v = load_f(y, y_dtype, yb + d);
    if (w != nullptr) v = v * r * (load_f(w, w_dtype, d) + plus_one);
    const float h = residual[rb + d] + mult * v;
    residual[rb + d] = h;
    if (out != nullptr) store_f(out, out_dtype, rb + d, h);
  }
}

// The same with the element types known at compile time and a row held in registers (NP elements a thread): every
// load of a row is asked for before the first use, so the kernel waits for memory once.  It runs a dozen times per
// layer and decode step on a handful of rows, where the kernel above, whose loads sit behind tests of the element
// type, took 10 us.
template <typename YT, typename WT, typename OT, int NP>
__global__ __launch_bounds__(256) void residual_add_norm_typed_kernel(
    const YT* __restrict__ y, int64_t y_stride, const WT* __restrict__ w, float eps, float plus_one, float mult,
    float* __restrict__ residual, OT* __restrict__ out, int D) {
  __shared__ float scratch[16];
  const size_t yb = static_cast<size_t>(blockIdx.x) * y_stride, rb = static_cast<size_t>(blockIdx.x) * D;
  float yv[NP], hv[NP], wv[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = threadIdx.x + p * 256;
    const bool ok = d < D;
    yv[p] = ok ? to_float(y[yb + d]) : 0.f;
    hv[p] = ok ? residual[rb + d] : 0.f;
    wv[p] = (ok && w != nullptr) ? to_float(w[d]) + plus_one : 1.f;
  }
  float r = 1.f;
  if (w != nullptr) {
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) ss = fmaf(yv[p], yv[p], ss);
    ss = block_sum(ss, scratch);
    r = 1.f / sqrtf(ss / static_cast<float>(D) + eps);
  }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = threadIdx.x + p * 256;
    if (d >= D) continue;
    const float v = w != nullptr ? yv[p] * r * wv[p] : yv[p];
    const float h = hv[p] + mult * v;
    residual[rb + d] = h;
    if (out != nullptr) out[rb + d] = from_float<OT>(h);
  }
}

// The same for rows in pieces of eight.
template <typename YT, typename WT, typename OT, int NP>
__global__ __launch_bounds__(256) void residual_add_norm_eights_kernel(
    const YT* __restrict__ y, int64_t y_stride, const WT* __restrict__ w, float eps, float plus_one, float mult,
    float* __restrict__ residual, OT* __restrict__ out, int D) {
  __shared__ float scratch[16];
  const YT* yr = y + static_cast<size_t>(blockIdx.x) * y_stride;
  const size_t rb = static_cast<size_t>(blockIdx.x) * D;
  Eight yv[NP], hv[NP], wv[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int at = (p * 256 + threadIdx.x) * 8, d = at < D ? at : D - 8;
    yv[p] = load_eight(yr + d);
    hv[p] = load_eight(residual + rb + d);
    if (w != nullptr) wv[p] = load_eight(w + d);
  }
  float r = 1.f;
  if (w != nullptr) {
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      float part = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) part = fmaf(yv[p].v[e], yv[p].v[e], part);
      ss += (p * 256 + threadIdx.x) * 8 < D ? part : 0.f;
    }
    ss = block_sum(ss, scratch);
    r = 1.f / sqrtf(ss / static_cast<float>(D) + eps);
  }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = (p * 256 + threadIdx.x) * 8;
    if (d >= D) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = w != nullptr ? yv[p].v[e] * r * (wv[p].v[e] + plus_one) : yv[p].v[e];
      hv[p].v[e] += mult * v;
    }
    store_eight(residual + rb + d, hv[p]);
    if (out != nullptr) store_eight(out + rb + d, hv[p]);
  }
}

template <typename YT, typename WT, typename OT>
static bool launch_residual_add_norm_typed(const void* y, int64_t y_stride, const void* w, float eps, float plus_one,
                                           float mult, float* residual, void* out, int T, int D, hipStream_t stream) {
  const YT* yp = static_cast<const YT*>(y);
  const WT* wp = static_cast<const WT*>(w);
  OT* op = static_cast<OT*>(out);
  if (D <= 8192 && rows_in_eights(D, y_stride, y, w, residual, out, nullptr)) {
    if (D <= 2048)
      residual_add_norm_eights_kernel<YT, WT, OT, 1><<<T, 256, 0, stream>>>(yp, y_stride, wp, eps, plus_one, mult, residual, op, D);
    else if (D <= 4096)
      residual_add_norm_eights_kernel<YT, WT, OT, 2><<<T, 256, 0, stream>>>(yp, y_stride, wp, eps, plus_one, mult, residual, op, D);
    else
      residual_add_norm_eights_kernel<YT, WT, OT, 4><<<T, 256, 0, stream>>>(yp, y_stride, wp, eps, plus_one, mult, residual, op, D);
    return true;
  }
  if (D <= 1024)
    residual_add_norm_typed_kernel<YT, WT, OT, 4><<<T, 256, 0, stream>>>(yp, y_stride, wp, eps, plus_one, mult, residual, op, D);
  else if (D <= 2048)
    residual_add_norm_typed_kernel<YT, WT, OT, 8><<<T, 256, 0, stream>>>(yp, y_stride, wp, eps, plus_one, mult, residual, op, D);
  else if (D <= 4096)
    residual_add_norm_typed_kernel<YT, WT, OT, 16><<<T, 256, 0, stream>>>(yp, y_stride, wp, eps, plus_one, mult, residual, op, D);
  else
    return false;
  return true;
}

// ------------------------------------------------------------------ residual += mult * y; out = norm(residual)
// The sum of a block that norms what its parts read (their results are added as they are, times a constant), fused
// with the norm in front of the next part: out = h / sqrt(mean(h^2) + eps) * (w + plus_one) over the updated row h,
// which is held in registers between the two.  y null: nothing is added.  CENTERED: a layer norm instead, out =
// (h - mean) / sqrt(mean((h - mean)^2) + eps) * (w + plus_one) + b.  A y_stride of 0 adds the same row to every row.
// The layer norm's mean and sum of squared deviations come from every wave's own, merged by the counts (one exchange
// through LDS, no cancellation).
template <typename YT, typename WT, typename OT, int NP, bool CENTERED>
__global__ __launch_bounds__(256) void residual_add_next_norm_kernel(
    const YT* __restrict__ y, int64_t y_stride, float mult, float* __restrict__ residual, const WT* __restrict__ w,
    const WT* __restrict__ b, float eps, float plus_one, OT* __restrict__ out, int D) {
  __shared__ float scratch[16];
  const size_t yb = static_cast<size_t>(blockIdx.x) * y_stride, rb = static_cast<size_t>(blockIdx.x) * D;
  float yv[NP], hv[NP], wv[NP], bv[CENTERED ? NP : 1];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = threadIdx.x + p * 256;
    const bool ok = d < D;
    yv[p] = (ok && y != nullptr) ? to_float(y[yb + d]) : 0.f;
    hv[p] = ok ? residual[rb + d] : 0.f;
    wv[p] = ok ? to_float(w[d]) + plus_one : 0.f;
    if constexpr (CENTERED) bv[p] = ok ? to_float(b[d]) : 0.f;
  }
  float ss = 0.f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = threadIdx.x + p * 256;
    if (y != nullptr) {
      hv[p] = hv[p] + mult * yv[p];
      if (d < D) residual[rb + d] = hv[p];
    }
    if constexpr (CENTERED) ss += hv[p];   // (entries beyond the row are zero)
    else ss = fmaf(hv[p], hv[p], ss);
  }
  if constexpr (CENTERED) {
    const int wave = threadIdx.x / kWave;
    int mine = 0;   // entries of the row that this wave holds
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int left = D - p * 256 - wave * kWave;
      mine += left < 0 ? 0 : left > kWave ? kWave : left;
    }
    const float part = mine > 0 ? wave_sum(ss) / static_cast<float>(mine) : 0.f;
    float sq = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const float e = hv[p] - part;
      if (threadIdx.x + p * 256 < D) sq = fmaf(e, e, sq);
    }
    sq = wave_sum(sq);
    if (threadIdx.x % kWave == 0) {
      scratch[wave] = part;
      scratch[4 + wave] = sq;
      scratch[8 + wave] = static_cast<float>(mine);
    }
    __syncthreads();
    float mean = 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v) mean = fmaf(scratch[v], scratch[8 + v], mean);
    mean /= static_cast<float>(D);
    ss = 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float e = scratch[v] - mean;
      ss += fmaf(e * e, scratch[8 + v], scratch[4 + v]);
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) hv[p] -= mean;
  } else {
    ss = block_sum(ss, scratch);
  }
  const float r = 1.f / sqrtf(ss / static_cast<float>(D) + eps);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = threadIdx.x + p * 256;
    if (d < D) out[rb + d] = from_float<OT>(CENTERED ? fmaf(hv[p] * r, wv[p], bv[CENTERED ? p : 0]) : hv[p] * r * wv[p]);
  }
}

// What is added to the residual, eight entries at a time: rows as they are ...
template <typename YT>
struct RowsAsTheyAre {
  const YT* y;
  int64_t stride;
  __device__ __forceinline__ Eight at(int row, int d) const { return load_eight(y + static_cast<size_t>(row) * stride + d); }
};
// ... or a token's experts' rows [tokens * top, D], weighted and added up in the order of its choices, and its shared row, times
// sigmoid(gate) if there is one: the sum over experts without a launch and a round trip of its own (8 tokens of
// 2,048: 4.8 + 4.6 us before, 4.8 now; 2,047 tokens 9.9 + 10.8 and 15.8).
template <typename ST>
struct RowsOfExperts {
  const float *y, *weights;
  const ST* shared;
  const float* gate;
  int64_t shared_stride, gate_stride;
  int top, D;
  __device__ __forceinline__ Eight at(int row, int d) const {
    Eight s;
#pragma unroll
    for (int e = 0; e < 8; ++e) s.v[e] = 0.f;
    if (shared != nullptr) s = load_eight(shared + static_cast<size_t>(row) * shared_stride + d);   // (asked for first)
    const float* from = y + static_cast<size_t>(row) * top * D + d;
    const float* w = weights + static_cast<size_t>(row) * top;
    Eight v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v.v[e] = 0.f;
#pragma unroll 2
    for (int k = 0; k < top; ++k) {
      const Eight q = load_eight(from + static_cast<size_t>(k) * D);
      const float wk = w[k];
#pragma unroll
      for (int e = 0; e < 8; ++e) v.v[e] = fmaf(wk, q.v[e], v.v[e]);
    }
    if (shared != nullptr) {
      const float f = gate != nullptr ? 1.f + expf(-gate[static_cast<size_t>(row) * gate_stride]) : 1.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) v.v[e] += gate != nullptr ? s.v[e] / f : s.v[e];
    }
    return v;
  }
};

// What becomes of the normed row: it goes to `out` as it is ...
struct RowItself {
  static constexpr int STREAMS = 0;
  __device__ __forceinline__ int meta(int, int) const { return 0; }
};
// ... or, in a step with one token of every request, only the mixes with the row before it that token_shift_kernel makes (the row
// rounded to bfloat16 first, as that kernel reads it), and the row becomes the request's last: a launch and a round trip less
// (8 tokens of 2,048 wide, five mixes: 4.7 + 5.1 us before, 4.8 now).
// Workgroup j has request j.
template <typename MT>
struct RowMixed {
  static constexpr int STREAMS = 5;
  const MT* mu;
  float* tails;
  int64_t tail_stride;
  const int* seq_meta;
  __device__ __forceinline__ int meta(int j, int i) const { return seq_meta[4 * j + i]; }
};

// The same for rows in pieces of eight (ADD: there is something to add).
template <typename SRC, typename WT, typename OT, int NP, bool CENTERED, bool ADD, typename TO = RowItself>
__global__ __launch_bounds__(256) void residual_add_next_norm_eights_kernel(
    SRC y, float mult, float* __restrict__ residual, const WT* __restrict__ w, const WT* __restrict__ b, float eps,
    float plus_one, OT* __restrict__ out, int D, TO to) {
  __shared__ float scratch[16];
  constexpr int STREAMS = TO::STREAMS;
  const int row = STREAMS > 0 ? to.meta(blockIdx.x, 1) : blockIdx.x;
  const size_t rb = static_cast<size_t>(row) * D;
  Eight yv[ADD ? NP : 1], hv[NP], wv[NP], bv[CENTERED ? NP : 1];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int at = (p * 256 + threadIdx.x) * 8, d = at < D ? at : D - 8;
    hv[p] = load_eight(residual + rb + d);
    wv[p] = load_eight(w + d);
    if constexpr (CENTERED) bv[p] = load_eight(b + d);
    if constexpr (ADD) yv[p] = y.at(row, d);
  }
  Eight before[STREAMS > 0 ? NP : 1], mix[STREAMS > 0 ? NP : 1][STREAMS > 0 ? STREAMS : 1];   // (asked for ahead of the sums)
  if constexpr (STREAMS > 0) {
    const float* tail = to.tails + static_cast<size_t>(to.meta(blockIdx.x, 0)) * to.tail_stride;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int at = (p * 256 + threadIdx.x) * 8, d = at < D ? at : D - 8;
      before[p] = load_eight(tail + d);
#pragma unroll
      for (int s = 0; s < STREAMS; ++s) mix[p][s] = load_eight(to.mu + static_cast<size_t>(s) * D + d);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = (p * 256 + threadIdx.x) * 8;
    if constexpr (ADD) {
#pragma unroll
      for (int e = 0; e < 8; ++e) hv[p].v[e] += mult * yv[p].v[e];
      if (d < D) store_eight(residual + rb + d, hv[p]);
    }
    float part = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) part = CENTERED ? part + hv[p].v[e] : fmaf(hv[p].v[e], hv[p].v[e], part);
    ss += d < D ? part : 0.f;
  }
  float mean = 0.f;
  if constexpr (CENTERED) {
    const int wave = threadIdx.x / kWave;
    int mine = 0;   // entries of the row that this wave holds
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int left = D - (p * 256 + wave * kWave) * 8;
      mine += left < 0 ? 0 : left > kWave * 8 ? kWave * 8 : left;
    }
    const float part = mine > 0 ? wave_sum(ss) / static_cast<float>(mine) : 0.f;
    float sq = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      float q = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = hv[p].v[e] - part;
        q = fmaf(x, x, q);
      }
      sq += (p * 256 + threadIdx.x) * 8 < D ? q : 0.f;
    }
    sq = wave_sum(sq);
    if (threadIdx.x % kWave == 0) {
      scratch[wave] = part;
      scratch[4 + wave] = sq;
      scratch[8 + wave] = static_cast<float>(mine);
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) mean = fmaf(scratch[v], scratch[8 + v], mean);
    mean /= static_cast<float>(D);
    ss = 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float e = scratch[v] - mean;
      ss += fmaf(e * e, scratch[8 + v], scratch[4 + v]);
    }
  } else {
    ss = block_sum(ss, scratch);
  }
  const float r = 1.f / sqrtf(ss / static_cast<float>(D) + eps);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int d = (p * 256 + threadIdx.x) * 8;
    if (d >= D) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float gain = wv[p].v[e] + plus_one;
      hv[p].v[e] = CENTERED ? fmaf((hv[p].v[e] - mean) * r, gain, bv[CENTERED ? p : 0].v[e]) : hv[p].v[e] * r * gain;
    }
    if constexpr (STREAMS > 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) hv[p].v[e] = to_float(from_float<OT>(hv[p].v[e]));
      store_eight(to.tails + static_cast<size_t>(to.meta(blockIdx.x, 0)) * to.tail_stride + d, hv[p]);
#pragma unroll
      for (int s = 0; s < STREAMS; ++s) {
        Eight v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v.v[e] = fmaf(before[p].v[e] - hv[p].v[e], mix[p][s].v[e], hv[p].v[e]);
        store_eight(out + rb * STREAMS + static_cast<size_t>(s) * D + d, v);
      }
    } else {
      store_eight(out + rb + d, hv[p]);
    }
  }
}

template <typename YT, typename WT, typename OT, bool CENTERED>
static void launch_residual_add_next_norm(const void* y, int64_t y_stride, float mult, float* residual, const void* w,
                                          const void* b, float eps, float plus_one, void* out, int T, int D,
                                          hipStream_t stream) {
  const RowsAsTheyAre<YT> rows{static_cast<const YT*>(y), y_stride};
#define SA_NEXT_NORM_EIGHTS(NP, ADD)                                                                                    \
  residual_add_next_norm_eights_kernel<RowsAsTheyAre<YT>, WT, OT, NP, CENTERED, ADD><<<T, 256, 0, stream>>>(            \
      rows, mult, residual, static_cast<const WT*>(w), static_cast<const WT*>(b), eps, plus_one, static_cast<OT*>(out), D, RowItself{})
  if (rows_in_eights(D, y != nullptr ? y_stride : 0, y, w, b, residual, out)) {
    if (y != nullptr) {
      if (D <= 2048) SA_NEXT_NORM_EIGHTS(1, true);
      else if (D <= 4096) SA_NEXT_NORM_EIGHTS(2, true);
      else SA_NEXT_NORM_EIGHTS(4, true);
    } else {
      if (D <= 2048) SA_NEXT_NORM_EIGHTS(1, false);
      else if (D <= 4096) SA_NEXT_NORM_EIGHTS(2, false);
      else SA_NEXT_NORM_EIGHTS(4, false);
    }
    return;
  }
#undef SA_NEXT_NORM_EIGHTS
#define SA_NEXT_NORM_NP(NP)                                                                                        \
  residual_add_next_norm_kernel<YT, WT, OT, NP, CENTERED><<<T, 256, 0, stream>>>(                                    \
      static_cast<const YT*>(y), y_stride, mult, residual, static_cast<const WT*>(w), static_cast<const WT*>(b), eps, \
      plus_one, static_cast<OT*>(out), D)
  if (D <= 1024) SA_NEXT_NORM_NP(4);
  else if (D <= 2048) SA_NEXT_NORM_NP(8);
  else if (D <= 4096) SA_NEXT_NORM_NP(16);
  else SA_NEXT_NORM_NP(32);
#undef SA_NEXT_NORM_NP
}

// ------------------------------------------------------------------ heads normed and gated
// out[t, h, :] = (w ? x[t, h, :] / sqrt(mean(x[t, h, :]^2) + eps) * w : x[t, h, :]) * gate(g[t, h, :]),
// gate 0: sigmoid, 1: silu.  One wave per (token, head); w [size] is shared by the heads, or (w_per_head) [H * size].
__device__ inline float gate_value(int kind, float g) {
  const float s = 1.f / (1.f + expf(-g));
  return kind == 1 ? g * s : s;
}

__global__ __launch_bounds__(kWave) void gated_heads_kernel(
    const void* __restrict__ x, int x_dtype, int64_t x_stride, const void* __restrict__ g, int g_dtype,
    int64_t g_stride, const void* __restrict__ w, int w_dtype, float eps, int gate, void* __restrict__ out,
    int out_dtype, int64_t out_stride, int size, int gate_per_head, int w_per_head) {
  // gate_per_head: a gate row holds one number per head, which all of the head's entries share
  const int t = blockIdx.x, h = blockIdx.y;
  const size_t xb = static_cast<size_t>(t) * x_stride + static_cast<size_t>(h) * size;
  const size_t gb = static_cast<size_t>(t) * g_stride + (gate_per_head ? h : static_cast<size_t>(h) * size);
  const size_t ob = static_cast<size_t>(t) * out_stride + static_cast<size_t>(h) * size;
  float r = 1.f;
  if (w != nullptr) {
    float ss = 0.f;
    for (int d = threadIdx.x; d < size; d += kWave) {
      const float v = load_f(x, x_dtype, xb + d);
      ss = fmaf(v, v, ss);
    }
    ss = wave_sum(ss);
    r = 1.f / sqrtf(ss / static_cast<float>(size) + eps);
  }
  for (int d = threadIdx.x; d < size; d += kWave) {
    float v = load_f(x, x_dtype, xb + d);
    if (w != nullptr) v = v * r * load_f(w, w_dtype, w_per_head ? static_cast<size_t>(h) * size + d : d);
    store_f(out, out_dtype, ob + d, v * gate_value(gate, load_f(g, g_dtype, gate_per_head ? gb : gb + d)));
  }
}

// The same in pieces of eight entries a lane, `per` (4 to 64, a power of two) lanes a head: for heads of 32 to 512 entries,
// gates per entry and results in bfloat16, rows aligned to 16 bytes.  Bound by memory: 2,047 tokens of 16 heads of 128 in 32
// bits (33 MB) take 9.6 us; entry by entry with a wave a head they took 16.7.
template <typename XT, typename WT>
__global__ __launch_bounds__(256) void gated_heads_eights_kernel(
    const XT* __restrict__ x, int64_t x_stride, const bf16* __restrict__ g, int64_t g_stride, const WT* __restrict__ w, float eps,
    int gate, bf16* __restrict__ out, int64_t out_stride, int H, int per, int w_per_head, int64_t heads) {
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t head = item / per;
  if (head >= heads) return;   // (all lanes of a head together: 256 and a wave are multiples of `per`)
  const int64_t t = head / H;
  const int h = static_cast<int>(head - t * H), d = static_cast<int>(item % per) * 8, size = per * 8;
  Eight v = load_eight(x + t * x_stride + static_cast<int64_t>(h) * size + d);
  const Eight gv = load_eight(g + t * g_stride + static_cast<int64_t>(h) * size + d);
  if (w != nullptr) {
    const Eight wv = load_eight(w + (w_per_head ? h * size : 0) + d);
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(v.v[i], v.v[i], ss);
    for (int n = 1; n < per; n *= 2) ss += __shfl_xor(ss, n);
    const float r = 1.f / sqrtf(ss / static_cast<float>(size) + eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) v.v[i] = v.v[i] * r * wv.v[i];
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) v.v[i] *= gate_value(gate, gv.v[i]);
  store_eight(out + t * out_stride + static_cast<int64_t>(h) * size + d, v);
}

template <typename XT, typename WT>
static void launch_gated_heads_eights(const void* x, int64_t x_stride, const void* g, int64_t g_stride, const void* w, float eps,
                                      int gate, void* out, int64_t out_stride, int T, int H, int size, int w_per_head,
                                      hipStream_t stream) {
  const int per = size / 8;
  const int64_t heads = static_cast<int64_t>(T) * H;
  gated_heads_eights_kernel<XT, WT><<<static_cast<unsigned>((heads * per + 255) / 256), 256, 0, stream>>>(
      static_cast<const XT*>(x), x_stride, static_cast<const bf16*>(g), g_stride, static_cast<const WT*>(w), eps, gate,
      static_cast<bf16*>(out), out_stride, H, per, w_per_head, heads);
}

// ------------------------------------------------------------------ an activation in place
__global__ void activation_kernel(void* __restrict__ x, int dtype, int64_t stride, int N, int act) {
  const size_t rb = static_cast<size_t>(blockIdx.y) * stride;
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n < N) store_f(x, dtype, rb + n, gated_activation_exact(act, load_f(x, dtype, rb + n)));
}

// ------------------------------------------------------------------ queries and keys: partial rotation, unit RMS
// One wave per (token, head) of a fused projection row [H * dk queries | K * dk keys | K * dv values | ...].
//   q, k: the first rot_dims dimensions are rotated in pairs (i, i + rot_dims / 2) by position * inv_freq[i], the
//         others pass; then the head is divided by sqrt(mean(x^2) + eps) (eps < 0: left as it is).  Queries, times
//         q_mult (the scores' factor, for attention kernels that have none), go back in place, keys into the key pages.
//   v:    v <- (1 - lambda) v + lambda v_first (v_first null: v as it is), into the value pages (transposed).
constexpr int kQkPerLane = 8;  // key sizes up to 512
template <typename T>
__global__ __launch_bounds__(kWave) void qk_norm_rope_cache_write_kernel(
    T* __restrict__ proj, int64_t row_stride, const int* __restrict__ positions, const float* __restrict__ inv_freq,
    int rot_dims, float eps, float q_mult, const T* __restrict__ v_first, int64_t v_first_stride,
    const void* __restrict__ lambda,
    int lambda_dtype, const int64_t* __restrict__ slot_mapping, T* __restrict__ k_pages, T* __restrict__ v_pages,
    int H, int K, int dk, int dv, int page_size) {
  const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  T* row = proj + static_cast<size_t>(t) * row_stride;
  if (head < H + K) {
    const bool is_q = head < H;
    T* src = row + static_cast<size_t>(head) * dk;
    const int half = rot_dims / 2;
    const float pos = static_cast<float>(positions[t]);
    float o[kQkPerLane];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < kQkPerLane; ++j) {
      const int i = lane + j * kWave;
      o[j] = 0.f;
      if (i < dk) {
        float v = to_float(src[i]);
        if (i < rot_dims) {
          const int pair = i < half ? i : i - half;
          float s, c;
          sincosf(pos * inv_freq[pair], &s, &c);
          const float other = to_float(src[i < half ? i + half : i - half]);
          v = i < half ? v * c - other * s : v * c + other * s;
        }
        o[j] = v;
        ss = fmaf(v, v, ss);
      }
    }
    ss = wave_sum(ss);
    const float r = eps >= 0.f ? 1.f / sqrtf(ss / static_cast<float>(dk) + eps) : 1.f;
    // (every lane has read what it needs of the head before any lane writes: the wave runs in lockstep, and the
    // reduction above lies between the reads and the writes)
    if (is_q) {
#pragma unroll
      for (int j = 0; j < kQkPerLane; ++j) {
        const int i = lane + j * kWave;
        if (i < dk) src[i] = from_float<T>(o[j] * r * q_mult);
      }
      return;
    }
    if (k_pages == nullptr) return;
    const int64_t slot = slot_mapping[t];
    if (slot < 0) return;
    const int koff = static_cast<int>(slot % page_size);
    T* dst = k_pages + ((slot / page_size) * K + (head - H)) * page_size * dk;
    const bool tiled = keys_tiled(page_size, dk);
#pragma unroll
    for (int j = 0; j < kQkPerLane; ++j) {
      const int i = lane + j * kWave;
      if (i < dk) dst[key_index(tiled, page_size, dk, koff, i)] = from_float<T>(o[j] * r);
    }
    return;
  }
  if (v_pages == nullptr) return;
  const int64_t slot = slot_mapping[t];
  if (slot < 0) return;
  const int vh = head - H - K;
  const T* src = row + static_cast<size_t>(H + K) * dk + static_cast<size_t>(vh) * dv;
  const T* first = v_first == nullptr ? nullptr : v_first + static_cast<size_t>(t) * v_first_stride + static_cast<size_t>(vh) * dv;
  const float lam = first != nullptr ? load_f(lambda, lambda_dtype, 0) : 0.f;
  // value pages are [page, head, dv, page_size]: the keys of a page are contiguous for each dimension
  T* dst = v_pages + ((slot / page_size) * K + vh) * page_size * dv + slot % page_size;
  for (int i = lane; i < dv; i += kWave) {
    float v = to_float(src[i]);
    if (first != nullptr) v = (1.f - lam) * v + lam * to_float(first[i]);
    dst[static_cast<size_t>(i) * page_size] = from_float<T>(v);
  }
}

// ------------------------------------------------------------------ queries and keys: weighted norm, then rotation
// One wave per (token, head) of a fused projection row [H * dk queries | K * dk keys | K * dv values | ...].  A query
// or key vector of dk entries is cut into `sub` equal parts (the score maps of a head); in every part
//   the first norm_dims entries are divided by sqrt(mean of their squares + eps) and multiplied by w[i] (w null: not),
//   then the entries [rot_at, rot_at + rot_dims) turn in neighbouring pairs: (u, v) at the pair p becomes
//   rot_mult * (u cos a - v sin a, v cos a + u sin a) with a = position * freq[p].
// Queries go back in place, keys into the key pages (rows of dk entries), values as they are into the value pages
// (transposed); dv == 0: there are no values.  norm_dims, rot_at and w are given for queries and for keys.
struct HeadNormRope {
  const void* w;
  int norm_dims, rot_at;
};
constexpr int kPartPerLane = 16;  // parts of up to 1024 entries
// NP: pieces of 64 entries that a lane holds of a part (registers for no more than the part needs)
template <typename T, int NP>
__global__ __launch_bounds__(kWave) void norm_rope_cache_write_kernel(
    T* __restrict__ proj, int64_t row_stride, const int* __restrict__ positions, const float* __restrict__ freq,
    int rot_dims, float rot_mult, HeadNormRope qn, HeadNormRope kn, int w_dtype, float eps, int sub,
    const int64_t* __restrict__ slot_mapping, T* __restrict__ k_pages, T* __restrict__ v_pages, int H, int K, int dk,
    int dv, int page_size, int key_values) {
  // key_values > 0: a key row's first key_values entries, as they are stored, are the token's values as well (a latent
  // that is scored and read): they also go into value pages [num_pages, K, key_values, page_size]
  const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  T* row = proj + static_cast<size_t>(t) * row_stride;
  if (head < H + K) {
    const bool is_q = head < H;
    const HeadNormRope hn = is_q ? qn : kn;
    const int ds = dk / sub;
    const float pos = static_cast<float>(positions[t]);
    int64_t slot = -1;
    T* dst = nullptr;
    bool tiled = false;
    int koff = 0;
    if (!is_q) {
      if (k_pages == nullptr) return;
      slot = slot_mapping[t];
      if (slot < 0) return;
      koff = static_cast<int>(slot % page_size);
      dst = k_pages + ((slot / page_size) * K + (head - H)) * page_size * dk;
      tiled = keys_tiled(page_size, dk);
    }
    for (int part = 0; part < sub; ++part) {
      T* src = row + static_cast<size_t>(head) * dk + static_cast<size_t>(part) * ds;
      float raw[NP], other[NP];
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const int i = lane + j * kWave;
        raw[j] = other[j] = 0.f;
        if (j * kWave < ds && i < ds) {   // (the first test is uniform: pieces beyond the part cost a branch)
          const int e = i - hn.rot_at;
          const bool turns = e >= 0 && e < rot_dims;
          // a query entry that is neither normed nor rotated stays where it is: it is not even read
          if (!is_q || turns || (hn.w != nullptr && i < hn.norm_dims)) raw[j] = to_float(src[i]);
          if (turns) other[j] = to_float(src[hn.rot_at + (e ^ 1)]);
          if (i < hn.norm_dims) ss = fmaf(raw[j], raw[j], ss);
        }
      }
      float r = 1.f;
      if (hn.w != nullptr && hn.norm_dims > 0) {
        ss = wave_sum(ss);
        r = 1.f / sqrtf(ss / static_cast<float>(hn.norm_dims) + eps);
      }
      // (every lane has read what it needs of the part before any lane writes: the wave runs in lockstep)
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const int i = lane + j * kWave;
        if (j * kWave >= ds || i >= ds) continue;
        if (is_q && (i - hn.rot_at < 0 || i - hn.rot_at >= rot_dims) && !(hn.w != nullptr && i < hn.norm_dims)) continue;
        float v = raw[j];
        if (hn.w != nullptr && i < hn.norm_dims) v = v * r * load_f(hn.w, w_dtype, i);
        const int e = i - hn.rot_at;
        if (e >= 0 && e < rot_dims) {
          const int pi = hn.rot_at + (e ^ 1);
          float o = other[j];
          if (hn.w != nullptr && pi < hn.norm_dims) o = o * r * load_f(hn.w, w_dtype, pi);
          float sn, cs;
          sincosf(pos * freq[e >> 1], &sn, &cs);
          sn *= rot_mult;
          cs *= rot_mult;
          v = (e & 1) == 0 ? v * cs - o * sn : v * cs + o * sn;
        }
        if (is_q) {
          src[i] = from_float<T>(v);
        } else {
          dst[key_index(tiled, page_size, dk, koff, part * ds + i)] = from_float<T>(v);
          if (part * ds + i < key_values)
            v_pages[(((slot / page_size) * K + (head - H)) * key_values + part * ds + i) * page_size + koff] =
                from_float<T>(v);
        }
      }
    }
    return;
  }
  if (v_pages == nullptr) return;
  const int64_t slot = slot_mapping[t];
  if (slot < 0) return;
  const int vh = head - H - K;
  const T* src = row + static_cast<size_t>(H + K) * dk + static_cast<size_t>(vh) * dv;
  T* dst = v_pages + ((slot / page_size) * K + vh) * page_size * dv + slot % page_size;
  for (int i = lane; i < dv; i += kWave) dst[static_cast<size_t>(i) * page_size] = src[i];
}

}  // namespace sa

using namespace sa;

extern "C" int sa_residual_add_norm(const void* y, int y_dtype, int64_t y_stride, const void* w, int w_dtype, float eps,
                                    int plus_one, float mult, float* residual, void* out, int out_dtype, int T, int D,
                                    hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && D > 0 && residual != nullptr, "residual_add_norm: bad sizes T=%d D=%d", T, D);
  SA_REQUIRE(y != nullptr || out != nullptr, "residual_add_norm: nothing to add and nowhere to hand the residual on");
  SA_REQUIRE(y == nullptr || y_stride == 0 || y_stride >= D, "residual_add_norm: row stride %lld is below the width %d",
             (long long)y_stride, D);
  SA_REQUIRE(eps >= 0.f, "residual_add_norm: eps must not be negative");
  // the usual combinations of element types have kernels of their own (a bfloat16 run, a 32-bit run)
  const float plus = plus_one ? 1.f : 0.f;
  bool done = false;
  if (y != nullptr && y_dtype == kBF16 && (w == nullptr || w_dtype == kBF16) && (out == nullptr || out_dtype == kBF16))
    done = launch_residual_add_norm_typed<bf16, bf16, bf16>(y, y_stride, w, eps, plus, mult, residual, out, T, D, stream);
  else if (y != nullptr && y_dtype == kF32 && (w == nullptr || w_dtype == kF32) && (out == nullptr || out_dtype == kF32))
    done = launch_residual_add_norm_typed<float, float, float>(y, y_stride, w, eps, plus, mult, residual, out, T, D, stream);
  if (!done)
    residual_add_norm_kernel<<<T, 256, 0, stream>>>(y, y_dtype, y_stride, w, w_dtype, eps, plus, mult, residual, out,
                                                    out_dtype, D);
  return check_launch("residual_add_norm");
}

extern "C" int sa_residual_add_next_norm(const void* y, int y_dtype, int64_t y_stride, float mult, float* residual,
                                         const void* w, const void* b, int w_dtype, float eps, int plus_one, void* out,
                                         int out_dtype, int T, int D, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && D > 0 && D <= 8192 && residual != nullptr && w != nullptr && out != nullptr,
             "residual_add_next_norm: bad sizes T=%d D=%d (rows of at most 8192), or a null pointer", T, D);
  SA_REQUIRE(y == nullptr || y_stride == 0 || y_stride >= D, "residual_add_next_norm: row stride %lld is below the width %d",
             (long long)y_stride, D);
  SA_REQUIRE(eps >= 0.f, "residual_add_next_norm: eps must not be negative");
  const float plus = plus_one ? 1.f : 0.f;
  const bool yb = y == nullptr ? out_dtype == kBF16 : y_dtype == kBF16;
  SA_REQUIRE((y == nullptr || y_dtype == kBF16 || y_dtype == kF32) && (out_dtype == kBF16 || out_dtype == kF32),
             "residual_add_next_norm: rows are bfloat16 or float32");
  SA_REQUIRE(w_dtype == kBF16 || w_dtype == kF32, "residual_add_next_norm: weights are bfloat16 or float32");
#define SA_NEXT_NORM_C(YT, WT, OT)                                                                                        \
  do {                                                                                                                    \
    if (b != nullptr)                                                                                                     \
      launch_residual_add_next_norm<YT, WT, OT, true>(y, y_stride, mult, residual, w, b, eps, plus, out, T, D, stream);   \
    else                                                                                                                  \
      launch_residual_add_next_norm<YT, WT, OT, false>(y, y_stride, mult, residual, w, b, eps, plus, out, T, D, stream);  \
  } while (0)
#define SA_NEXT_NORM(YT, OT)                               \
  do {                                                     \
    if (w_dtype == kBF16) SA_NEXT_NORM_C(YT, bf16, OT);    \
    else SA_NEXT_NORM_C(YT, float, OT);                    \
  } while (0)
  if (yb && out_dtype == kBF16) SA_NEXT_NORM(bf16, bf16);
  else if (yb) SA_NEXT_NORM(bf16, float);
  else if (out_dtype == kBF16) SA_NEXT_NORM(float, bf16);
  else SA_NEXT_NORM(float, float);
#undef SA_NEXT_NORM
#undef SA_NEXT_NORM_C
  return check_launch("residual_add_next_norm");
}

// A workgroup adds a token's rows up one after the other, four pieces of 2,048 entries with their own sums each; the sum's kernel has a
// workgroup per piece.  Fused / sum and norm in us, 1, 64 and 2,047 tokens: 2,048 wide, top 16 3.8 / 4.9, 6.0 / 6.9, 59 / 63; 4,096,
// top 8 4.6 / 5.2, 6.8 / 7.3, 69 / 72, top 16 5.8 / 5.6, 9.3 / 8.3, 125 / 130; 8,192, top 2 5.8 / 6.2, 7.9 / 8.2, 61 / 66, top 4
// 6.5 / 6.1, 9.0 / 8.7, 89 / 98, top 16 15.8 / 6.6, 27.9 / 15.2, 249 / 249.
extern "C" int sa_experts_add_next_norm_pays(int D, int top) { return top <= (D <= 2048 ? 16 : D <= 4096 ? 8 : 2); }

extern "C" int sa_experts_add_next_norm_takes(int D, const void* shared, int64_t shared_stride, const void* residual, const void* w,
                                              const void* b) {
  return D <= 8192 && rows_in_eights(D, shared != nullptr ? shared_stride : 0, shared, residual, w, b, nullptr);
}

extern "C" int sa_experts_add_next_norm(const float* y, const float* weights, int top, const void* shared, int shared_dtype,
                                        int64_t shared_stride, const float* gate, int64_t gate_stride, float mult, float* residual,
                                        const void* w, const void* b, int w_dtype, float eps, int plus_one, void* out, int T, int D,
                                        hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && D > 0 && top > 0 && y != nullptr && weights != nullptr && residual != nullptr && w != nullptr && out != nullptr &&
                 (shared == nullptr || shared_stride >= D),
             "experts_add_next_norm: bad sizes T=%d D=%d top=%d, or a null pointer", T, D, top);
  SA_REQUIRE(sa_experts_add_next_norm_takes(D, shared, shared_stride, residual, w, b) && rows_in_eights(D, 0, y, out, nullptr, nullptr, nullptr),
             "experts_add_next_norm: rows of %d are not whole aligned pieces of 8 entries (8192 at most)", D);
  SA_REQUIRE(eps >= 0.f, "experts_add_next_norm: eps must not be negative");
  SA_REQUIRE((w_dtype == kBF16 || w_dtype == kF32) && (shared == nullptr || shared_dtype == kF32 || shared_dtype == kBF16),
             "experts_add_next_norm: weights and shared rows are bfloat16 or float32");
  const float plus = plus_one ? 1.f : 0.f;
#define SA_EXPERTS_NORM_NP(ST, WT, NP, C)                                                                                  \
  residual_add_next_norm_eights_kernel<RowsOfExperts<ST>, WT, bf16, NP, C, true><<<T, 256, 0, stream>>>(                   \
      RowsOfExperts<ST>{y, weights, static_cast<const ST*>(shared), gate, shared_stride, gate_stride, top, D}, mult, residual, \
      static_cast<const WT*>(w), static_cast<const WT*>(b), eps, plus, static_cast<bf16*>(out), D, RowItself{})
#define SA_EXPERTS_NORM_C(ST, WT, C)                          \
  do {                                                        \
    if (D <= 2048) SA_EXPERTS_NORM_NP(ST, WT, 1, C);          \
    else if (D <= 4096) SA_EXPERTS_NORM_NP(ST, WT, 2, C);     \
    else SA_EXPERTS_NORM_NP(ST, WT, 4, C);                    \
  } while (0)
#define SA_EXPERTS_NORM(ST, WT)                           \
  do {                                                    \
    if (b != nullptr) SA_EXPERTS_NORM_C(ST, WT, true);    \
    else SA_EXPERTS_NORM_C(ST, WT, false);                \
  } while (0)
  const bool s32 = shared == nullptr || shared_dtype == kF32;
  if (s32 && w_dtype == kBF16) SA_EXPERTS_NORM(float, bf16);
  else if (s32) SA_EXPERTS_NORM(float, float);
  else if (w_dtype == kBF16) SA_EXPERTS_NORM(bf16, bf16);
  else SA_EXPERTS_NORM(bf16, float);
#undef SA_EXPERTS_NORM
#undef SA_EXPERTS_NORM_C
#undef SA_EXPERTS_NORM_NP
  return check_launch("experts_add_next_norm");
}

extern "C" int sa_add_next_norm_shift_takes(int D, int streams, const void* y, int64_t y_stride, const void* shared, int64_t shared_stride,
                                            const void* residual, const void* w, const void* b, const void* mu, const void* tails,
                                            int64_t tail_stride) {
  return streams == RowMixed<bf16>::STREAMS && D <= 4096 && tail_stride % 4 == 0 && rows_in_eights(D, y_stride, y, residual, w, b, mu) &&
         rows_in_eights(D, shared != nullptr ? shared_stride : 0, shared, tails, nullptr, nullptr, nullptr);
}

namespace sa {
template <typename SRC, bool ADD, typename WT>
static void launch_next_norm_shift(const SRC& y, float mult, float* residual, const void* w, const void* b, float eps, float plus,
                                   const RowMixed<WT>& to, void* out, int T, int D, hipStream_t stream) {
  const WT *wt = static_cast<const WT*>(w), *bt = static_cast<const WT*>(b);
  bf16* o = static_cast<bf16*>(out);
#define SA_SHIFT_NORM(NP, C) \
  residual_add_next_norm_eights_kernel<SRC, WT, bf16, NP, C, ADD, RowMixed<WT>><<<T, 256, 0, stream>>>(y, mult, residual, wt, bt, eps, plus, o, D, to)
  if (D <= 2048) {
    if (b != nullptr) SA_SHIFT_NORM(1, true);
    else SA_SHIFT_NORM(1, false);
  } else {
    if (b != nullptr) SA_SHIFT_NORM(2, true);
    else SA_SHIFT_NORM(2, false);
  }
#undef SA_SHIFT_NORM
}
}  // namespace sa

extern "C" int sa_add_next_norm_shift(const void* y, int64_t y_stride, const float* weights, int top, const void* shared, int shared_dtype,
                                      int64_t shared_stride, const float* gate, int64_t gate_stride, float mult, float* residual,
                                      const void* w, const void* b, int w_dtype, float eps, int plus_one, const void* mu, int streams,
                                      float* tails, int64_t tail_stride, const int* seq_meta, void* out, int T, int D, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && D > 0 && residual != nullptr && w != nullptr && mu != nullptr && tails != nullptr && seq_meta != nullptr && out != nullptr &&
                 (weights == nullptr || (y != nullptr && top > 0)) && (shared == nullptr || (weights != nullptr && shared_stride >= D)),
             "add_next_norm_shift: bad sizes T=%d D=%d top=%d, or a null pointer", T, D, top);
  SA_REQUIRE(tail_stride >= D && (weights != nullptr || y_stride == 0 || y_stride >= D), "add_next_norm_shift: rows are shorter than the width %d", D);
  SA_REQUIRE(sa_add_next_norm_shift_takes(D, streams, y, weights == nullptr && y != nullptr ? y_stride : 0, shared, shared_stride, residual, w, b, mu,
                                          tails, tail_stride) && rows_in_eights(D, 0, out, nullptr, nullptr, nullptr, nullptr),
             "add_next_norm_shift: rows of %d are not whole aligned pieces of 8 entries (4096 at most), or not 5 streams", D);
  SA_REQUIRE(eps >= 0.f, "add_next_norm_shift: eps must not be negative");
  SA_REQUIRE((w_dtype == kBF16 || w_dtype == kF32) && (shared == nullptr || shared_dtype == kF32 || shared_dtype == kBF16),
             "add_next_norm_shift: weights and shared rows are bfloat16 or float32");
  const float plus = plus_one ? 1.f : 0.f;
  const auto run = [&](auto one) {
    using WT = decltype(one);
    const RowMixed<WT> to{static_cast<const WT*>(mu), tails, tail_stride, seq_meta};
    const float* rows = static_cast<const float*>(y);
    if (weights == nullptr && y == nullptr)
      launch_next_norm_shift<RowsAsTheyAre<bf16>, false, WT>(RowsAsTheyAre<bf16>{}, mult, residual, w, b, eps, plus, to, out, T, D, stream);
    else if (weights == nullptr)
      launch_next_norm_shift<RowsAsTheyAre<bf16>, true, WT>(RowsAsTheyAre<bf16>{static_cast<const bf16*>(y), y_stride}, mult, residual, w, b,
                                                            eps, plus, to, out, T, D, stream);
    else if (shared == nullptr || shared_dtype == kF32)
      launch_next_norm_shift<RowsOfExperts<float>, true, WT>(
          RowsOfExperts<float>{rows, weights, static_cast<const float*>(shared), gate, shared_stride, gate_stride, top, D}, mult, residual, w, b,
          eps, plus, to, out, T, D, stream);
    else
      launch_next_norm_shift<RowsOfExperts<bf16>, true, WT>(
          RowsOfExperts<bf16>{rows, weights, static_cast<const bf16*>(shared), gate, shared_stride, gate_stride, top, D}, mult, residual, w, b,
          eps, plus, to, out, T, D, stream);
  };
  if (w_dtype == kBF16) run(bf16{});
  else run(float{});
  return check_launch("add_next_norm_shift");
}

extern "C" int sa_gated_heads(const void* x, int x_dtype, int64_t x_stride, const void* g, int g_dtype, int64_t g_stride,
                              const void* w, int w_dtype, float eps, int gate, void* out, int out_dtype,
                              int64_t out_stride, int T, int H, int size, int gate_per_head, int w_per_head,
                              hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && H > 0 && size > 0 && x != nullptr && g != nullptr && out != nullptr,
             "gated_heads: bad sizes T=%d H=%d size=%d", T, H, size);
  const int64_t width = static_cast<int64_t>(H) * size;
  SA_REQUIRE(x_stride >= width && g_stride >= (gate_per_head ? H : width) && out_stride >= width,
             "gated_heads: a row stride is below %lld", (long long)width);
  SA_REQUIRE(gate == 0 || gate == 1, "gated_heads: unknown gate %d (0: sigmoid, 1: silu)", gate);
  SA_REQUIRE(H <= 65535, "gated_heads: at most 65535 heads");
  const auto aligned = [](const void* p, int64_t stride, int dtype) {
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && stride % (dtype == kF32 ? 4 : 8) == 0;
  };
  const bool known = (x_dtype == kF32 || x_dtype == kBF16) && (w == nullptr || w_dtype == kF32 || w_dtype == kBF16);
  if (known && g_dtype == kBF16 && out_dtype == kBF16 && !gate_per_head && size >= 32 && size <= 512 && (size & (size - 1)) == 0 &&
      aligned(x, x_stride, x_dtype) && aligned(g, g_stride, kBF16) && aligned(out, out_stride, kBF16) &&
      aligned(w, 0, kBF16)) {
    if (x_dtype == kF32 && (w == nullptr || w_dtype == kBF16))
      launch_gated_heads_eights<float, bf16>(x, x_stride, g, g_stride, w, eps, gate, out, out_stride, T, H, size, w_per_head, stream);
    else if (x_dtype == kF32)
      launch_gated_heads_eights<float, float>(x, x_stride, g, g_stride, w, eps, gate, out, out_stride, T, H, size, w_per_head, stream);
    else if (w == nullptr || w_dtype == kBF16)
      launch_gated_heads_eights<bf16, bf16>(x, x_stride, g, g_stride, w, eps, gate, out, out_stride, T, H, size, w_per_head, stream);
    else
      launch_gated_heads_eights<bf16, float>(x, x_stride, g, g_stride, w, eps, gate, out, out_stride, T, H, size, w_per_head, stream);
    return check_launch("gated_heads");
  }
  gated_heads_kernel<<<dim3(T, H), kWave, 0, stream>>>(x, x_dtype, x_stride, g, g_dtype, g_stride, w, w_dtype, eps, gate,
                                                       out, out_dtype, out_stride, size, gate_per_head, w_per_head);
  return check_launch("gated_heads");
}

namespace sa {
int apply_activation(void* x, int dtype, int64_t stride, int M, int N, int act, hipStream_t stream) {
  return sa_activation(x, dtype, stride, M, N, act, stream);
}
}  // namespace sa

extern "C" int sa_activation(void* x, int dtype, int64_t stride, int T, int N, int act, hipStream_t stream) {
  if (T == 0 || N == 0) return 0;
  SA_REQUIRE(T > 0 && N > 0 && stride >= N && T <= 65535 * 1024, "activation: bad sizes T=%d N=%d", T, N);
  SA_REQUIRE(act >= 0 && act < kNumActivations, "activation: unknown activation %d", act);
  SA_REQUIRE(dtype == kF32 || dtype == kBF16, "activation: unknown dtype %d", dtype);
  // rows beyond 65535 go in further launches (the grid's second dimension)
  for (int t0 = 0; t0 < T; t0 += 65535) {
    const int rows = T - t0 < 65535 ? T - t0 : 65535;
    char* base = static_cast<char*>(x) + static_cast<size_t>(t0) * stride * (dtype == kF32 ? 4 : 2);
    activation_kernel<<<dim3((N + 255) / 256, rows), 256, 0, stream>>>(base, dtype, stride, N, act);
  }
  return check_launch("activation");
}

extern "C" int sa_qk_norm_rope_cache_write(void* proj, int dtype, int64_t row_stride, const int* positions,
                                           const float* inv_freq, int rot_dims, float eps, float q_mult,
                                           const void* v_first, int64_t v_first_stride, const void* lambda, int lambda_dtype,
                                           const int64_t* slot_mapping, void* k_pages, void* v_pages, int T, int H,
                                           int K, int dk, int dv, int page_size, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(T > 0 && H >= 0 && K >= 0 && H + 2 * K > 0 && dk > 0 && dv > 0 && page_size > 0,
             "qk_norm_rope_cache_write: bad sizes T=%d H=%d K=%d dk=%d dv=%d P=%d", T, H, K, dk, dv, page_size);
  SA_REQUIRE(dk <= kQkPerLane * kWave, "qk_norm_rope_cache_write: key size %d is above %d", dk, kQkPerLane * kWave);
  SA_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= dk && (rot_dims == 0 || inv_freq != nullptr),
             "qk_norm_rope_cache_write: %d rotated dimensions of %d (an even number, with their frequencies)", rot_dims, dk);
  SA_REQUIRE(row_stride >= static_cast<int64_t>(H + K) * dk + static_cast<int64_t>(K) * dv,
             "qk_norm_rope_cache_write: row stride %lld is too small", (long long)row_stride);
  SA_REQUIRE((k_pages == nullptr) == (v_pages == nullptr) && (k_pages == nullptr || slot_mapping != nullptr),
             "qk_norm_rope_cache_write: key pages, value pages and slots come together");
  SA_REQUIRE(v_first == nullptr || (lambda != nullptr && v_first_stride >= static_cast<int64_t>(K) * dv),
             "qk_norm_rope_cache_write: mixed values need the factor and rows of K * dv values");
  SA_REQUIRE(H + 2 * K <= 65535, "qk_norm_rope_cache_write: too many heads");
  const dim3 grid(T, H + 2 * K);
  if (dtype == kF32)
    qk_norm_rope_cache_write_kernel<float><<<grid, kWave, 0, stream>>>(
        static_cast<float*>(proj), row_stride, positions, inv_freq, rot_dims, eps, q_mult, static_cast<const float*>(v_first),
        v_first_stride, lambda, lambda_dtype, slot_mapping, static_cast<float*>(k_pages), static_cast<float*>(v_pages),
        H, K, dk, dv, page_size);
  else if (dtype == kBF16)
    qk_norm_rope_cache_write_kernel<bf16><<<grid, kWave, 0, stream>>>(
        static_cast<bf16*>(proj), row_stride, positions, inv_freq, rot_dims, eps, q_mult, static_cast<const bf16*>(v_first),
        v_first_stride, lambda, lambda_dtype, slot_mapping, static_cast<bf16*>(k_pages), static_cast<bf16*>(v_pages), H,
        K, dk, dv, page_size);
  else
    SA_REQUIRE(false, "qk_norm_rope_cache_write: unknown dtype %d", dtype);
  return check_launch("qk_norm_rope_cache_write");
}

extern "C" int sa_norm_rope_cache_write(void* proj, int dtype, int64_t row_stride, const int* positions,
                                        const float* freq, int rot_dims, float rot_mult, const void* q_weight,
                                        int q_norm_dims, int q_rot_at, const void* k_weight, int k_norm_dims,
                                        int k_rot_at, int w_dtype, float eps, int sub, const int64_t* slot_mapping,
                                        void* k_pages, void* v_pages, int T, int H, int K, int dk, int dv,
                                        int page_size, int key_values, hipStream_t stream) {
  if (T == 0) return 0;
  SA_REQUIRE(key_values >= 0 && key_values <= dk && (key_values == 0 || (dv == 0 && v_pages != nullptr)),
             "norm_rope_cache_write: %d of a key row's %d entries as values (then there are value pages and no values "
             "of their own)", key_values, dk);
  SA_REQUIRE(T > 0 && H >= 0 && K >= 0 && H + K > 0 && dk > 0 && dv >= 0 && page_size > 0 && sub > 0,
             "norm_rope_cache_write: bad sizes T=%d H=%d K=%d dk=%d dv=%d P=%d sub=%d", T, H, K, dk, dv, page_size, sub);
  SA_REQUIRE(dk % sub == 0 && dk / sub <= kPartPerLane * kWave,
             "norm_rope_cache_write: vectors of %d entries in %d parts (equal parts of at most %d)", dk, sub,
             kPartPerLane * kWave);
  const int ds = dk / sub;
  SA_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && (rot_dims == 0 || freq != nullptr) && q_rot_at >= 0 && k_rot_at >= 0 &&
                 q_rot_at + rot_dims <= ds && k_rot_at + rot_dims <= ds,
             "norm_rope_cache_write: %d rotated entries do not fit into parts of %d", rot_dims, ds);
  SA_REQUIRE(q_norm_dims >= 0 && q_norm_dims <= ds && k_norm_dims >= 0 && k_norm_dims <= ds && eps >= 0.f,
             "norm_rope_cache_write: normed entries beyond a part, or a negative eps");
  SA_REQUIRE(row_stride >= static_cast<int64_t>(H + K) * dk + static_cast<int64_t>(K) * dv,
             "norm_rope_cache_write: row stride %lld is too small", (long long)row_stride);
  SA_REQUIRE(k_pages == nullptr || (slot_mapping != nullptr && (dv == 0 || v_pages != nullptr)),
             "norm_rope_cache_write: key pages come with slots (and value pages, if there are values)");
  SA_REQUIRE(H + 2 * K <= 65535, "norm_rope_cache_write: too many heads");
  const dim3 grid(T, H + K + (dv > 0 ? K : 0));
  const HeadNormRope qn{q_weight, q_norm_dims, q_rot_at}, kn{k_weight, k_norm_dims, k_rot_at};
  SA_REQUIRE(dtype == kF32 || dtype == kBF16, "norm_rope_cache_write: unknown dtype %d", dtype);
#define SA_LAUNCH(NP)                                                                                                 \
  do {                                                                                                                \
    if (dtype == kF32)                                                                                                \
      norm_rope_cache_write_kernel<float, NP><<<grid, kWave, 0, stream>>>(                                            \
          static_cast<float*>(proj), row_stride, positions, freq, rot_dims, rot_mult, qn, kn, w_dtype, eps, sub,      \
          slot_mapping, static_cast<float*>(k_pages), static_cast<float*>(v_pages), H, K, dk, dv, page_size,          \
          key_values);                                                                                                \
    else                                                                                                              \
      norm_rope_cache_write_kernel<bf16, NP><<<grid, kWave, 0, stream>>>(                                             \
          static_cast<bf16*>(proj), row_stride, positions, freq, rot_dims, rot_mult, qn, kn, w_dtype, eps, sub,       \
          slot_mapping, static_cast<bf16*>(k_pages), static_cast<bf16*>(v_pages), H, K, dk, dv, page_size,            \
          key_values);                                                                                                \
  } while (0)
  const int pieces = (ds + kWave - 1) / kWave;
  if (pieces <= 1) SA_LAUNCH(1);
  else if (pieces <= 2) SA_LAUNCH(2);
  else if (pieces <= 4) SA_LAUNCH(4);
  else if (pieces <= 9) SA_LAUNCH(9);
  else SA_LAUNCH(16);
#undef SA_LAUNCH
  return check_launch("norm_rope_cache_write");
}
