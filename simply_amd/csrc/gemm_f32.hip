// C[M, N] = epilogue(A[M, K] . W[N, K]^T) in 32 bits on the matrix cores.  Row-major float operands whose rows are multiples of 16
// bytes; everything else of the 32-bit path goes to gemm_generic.hip.
//
// Two kinds of products, by K alone.  Where K is cut into segments of whole stages of 32 columns (multiples of 256, and other
// multiples of 32), every number is taken as the sum of three bfloat16 ones, which hold its 24 bits exactly, and a product as the six
// of them that matter, on v_mfma_f32_16x16x32_bf16: 417 TFLOP/s of whole products at the unit's nominal rate where the 32-bit unit
// has 157.  Sums are 32-bit in either case, and with the bfloat16 unit's fewer roundings (six for 32 columns where the 32-bit unit
// has eight) errors of a product against 64 bits are smaller, at every one of the sizes below (root mean square over the result's: 3.7e-7
// for 4.5e-7 gated, 5.2e-7 for 6.1e-7 at K = 9,216, 2.4e-7 for 2.9e-7 at 2,048), down to the smallest 32-bit numbers (see kScale).
// Elsewhere v_mfma_f32_16x16x4_f32.
//
// Every output element is summed in one order whatever M is, so a row's result does not depend on which other rows are in
// the batch: K is cut into at most eight segments of the same length, a multiple of 16 (the length depends on K alone); a
// segment is summed by one chain of instructions in increasing blocks (of 32 columns, smallest parts first; or of 16: k = j, 4 + j,
// 8 + j, 12 + j together for j = 0 .. 3), and the segments' sums are added in increasing order.  Three ways of running that:
//
//   few rows    (M <= 16) a workgroup owns 16 rows of W, a wave a segment of them: bound by reading W once.  Loads bring
//               whole 128-byte pieces of rows, two to four stages of 32 columns of K ahead in registers; the operand order is made
//               on the way through LDS (each wave its own part, no barrier in the loop; 16-byte pieces permuted by row, so
//               that neither side has bank conflicts).
//   tiles       a workgroup of two to eight waves owns a tile of outputs and walks through all segments, adding a segment's sum to
//               its total at the segment's end: bound by the matrix unit and, with parts, the power that it draws.
//   cut tiles   a workgroup per segment; a sum kernel adds the segments' planes: where the tiles alone leave CUs idle.  With parts
//               only the tiles behind the last 256 whole ones are cut.
//
// Products of parts whose sums are no finite numbers are done again on the 32-bit unit, in the workgroup that has them (see redo).  That
// takes, in us, without / one row / all rows of such: 4 rows against (9,216 gated, 2,304) 37 / 67 / 69, 509 rows 230 / 430 / 1,000, against
// (2,304, 9,216) 114 / 310 / 860; 4 rows against (256,000, 2,304) 390 / 850 / 820.
//
// Measured, us, weights from HBM; "unit" with the 32-bit matrix unit throughout (many launches in a row; clocks differ by 5 to 8 % from one
// run to the next):
//   (N, K)                 4 rows, unit   12, unit    17, unit    61, unit    509, unit      1,024, unit
//   (2304, 2048)           8.6, 8.3       9.2, 9.2    14.7, 15.0  15.6, 16.8  41, 54         73, 104
//   (2304, 9216)           24.2, 23.9     26.9, 26.0  41, 45      39, 45      122, 175       223, 333
//   (4096, 2304)           10.2, 9.6      10.2, 10.8  16.1, 17.0  17.4, 18.9  75, 86         107, 155
//   (9216 gated, 2304)     36.9, 43.7     39.5, 45.2  51, 58      57, 64      218, 329       405, 637 (215 TFLOP/s)
//   (3584, 14336)          39.4, 39.1     43.6, 43.4  61, 65      61, 67      265, 397       535, 873
//   (14336 gated, 3584)    79, 87         83, 88      95, 123     117, 127    496, 770       1,014, 1,528
//   (4608, 36864)          170, 166       195, 189    163, 222    203, 224    863, 1,244     1,702, 2,737
//   (36864 gated, 4608)    234, 242       241, 250    305, 381    316, 395    1,590, 2,502   3,047, 4,948
//   (256000, 2304)         393, 400 (6.0 TB/s)  478, 508  541, 650  555, 661  2,830, 4,390   5,490, 8,626
#include <type_traits>

#include "api.h"
#include "common.h"

namespace sa {
namespace f32 {

typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

constexpr int kSegments = 8;
constexpr int BK = 32;         // columns of K of a stage: a row of a tile is 128 bytes
constexpr int kPieces = BK / 4;

struct Args {
  const float* A;
  const float* W;
  const float* W2;
  float* C;
  int64_t lda, ldc;
  int M, N, K;
  int seg;      // length of a segment, a multiple of 16
  int act;
  float cap;
  bool parts;   // products of parts on the bfloat16 matrix unit
};

// Where the 16-byte piece p of row r lies in a tile of rows of 128 bytes (in floats).
__device__ __forceinline__ int piece_at(int r, int p) { return r * BK + ((p ^ (r & 7)) * 4); }

// Eight numbers, each as the sum of three bfloat16 ones, which hold its 24 bits exactly (see kScale): the first is the number rounded,
// the second what that leaves rounded, the third what both leave.
struct Parts {
  bf16x8 p[3];
};
// Two numbers rounded, in one register, and what that leaves of them, which is exact.  DOT: what is left by one instruction a number
// (3.5 in all for the three parts instead of 5.5), for kernels that the vector unit bounds (256,000 outputs of 4 rows: 378 us for
// 403); beside many matrix instructions it is the slower one (509 gated rows: 256 us for 244).
template <bool DOT = false>
__device__ __forceinline__ uint32_t round_two(float& a, float& b) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  typedef __attribute__((ext_vector_type(2))) float floatx2;
  uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{a, b}), bf16x2));
  if constexpr (DOT) {
    uint32_t first = 0x0000bf80u, second = 0xbf800000u;   // -1 for one of the two
    asm("" : "+s"(first));   // (in registers: as an operand of the instruction itself, -1 is not the first of a pair)
    asm("" : "+s"(second));
    const bf16x2 v = __builtin_bit_cast(bf16x2, u);
    a = __builtin_amdgcn_fdot2_f32_bf16(v, __builtin_bit_cast(bf16x2, first), a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(v, __builtin_bit_cast(bf16x2, second), b, false);
  } else {
    asm("" : "+v"(u));   // (hides where the bits come from: the compiler would round each number once more by itself)
    a -= __uint_as_float(u << 16);
    b -= __uint_as_float(u & 0xffff0000u);
  }
  return u;
}
template <bool DOT = false>
__device__ __forceinline__ Parts parts(floatx4 a, floatx4 b) {
  float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  Parts r;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    typedef __attribute__((ext_vector_type(4))) uint32_t uint32x4;
    uint32x4 u;
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = round_two<DOT>(v[2 * i], v[2 * i + 1]);
    r.p[q] = __builtin_bit_cast(bf16x8, u);
  }
  return r;
}
// The products of parts that a sum of K products takes, smallest first; the three that are left out are below 2^-26 of the number's
// product.
constexpr int kProducts = 6;
constexpr int kPartOfW[kProducts] = {2, 0, 1, 1, 0, 0}, kPartOfX[kProducts] = {0, 2, 1, 0, 1, 0};

// The bfloat16 unit drops what lies below a sum's last bits, towards minus infinity: 0.3 of the root mean square error of a sum of
// 9,216 products, the same way in every sum.  Every other segment is therefore summed with its sign turned.
__device__ __forceinline__ float segment_sign(int segment) { return segment % 2 ? -1.f : 1.f; }
// A bfloat16 ends at 2^-133, and below 2^-126 the unit drops more of a sum's bits: with parts as they come, a sum of numbers around 2^-116
// would be 2e-6 off, around 2^-126 2e-3.  Both factors are therefore taken 2^24 times as large, which leaves no bit of a 32-bit number,
// subnormal ones included, below 2^-126; sums are scaled back.  Numbers of 2^104 and more, and sums of 2^80 and more, become infinite.
constexpr float kScale = 16777216.f, kUnscale = 1.f / kScale / kScale;

__device__ __forceinline__ bool finite(float v) { return fabsf(v) <= 3.402823466e38f; }
template <int EPI>
__device__ __forceinline__ float finish(const Args& a, float x, float y) {
  if (EPI == 1) return gated_product_exact(a.act, a.cap, x, y);
  if (EPI == 2) return a.cap * tanhf(x / a.cap);
  return x;
}

__device__ __forceinline__ void store4(const Args& a, int m, int n, floatx4 v) {
  float* dst = a.C + static_cast<size_t>(m) * a.ldc + n;
  if (n + 3 < a.N && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
    *reinterpret_cast<floatx4*>(dst) = v;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < a.N) dst[r] = v[r];
  }
}

// Sums of NB blocks of 16 weight rows (w: lane c's row of each, from its columns 4 g on) with 16 rows (x likewise), over the columns from
// k0 to k1, on the 32-bit matrix unit and in this file's order for it, added to `total`.
template <int NB>
__device__ __forceinline__ void plain_segment(const float* x, const float* const (&w)[NB], int k0, int k1, floatx4 (&total)[NB]) {
  floatx4 acc[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int k = k0; k < k1; k += 16) {
    const floatx4 xv = *reinterpret_cast<const floatx4*>(x + k);
    floatx4 wv[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) wv[t] = *reinterpret_cast<const floatx4*>(w[t] + k);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < NB; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t][j], xv[j], acc[t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < NB; ++t) total[t] += acc[t];
}
// Where the numbers of row m of A (of output n's weights) begin that lane group g multiplies; behind the last: the last.
__device__ __forceinline__ const float* row_of(const float* rows, int64_t stride, int i, int count, int g) {
  return rows + static_cast<size_t>(i < count ? i : count - 1) * stride + 4 * g;
}

// Products of parts give no finite number where a part is infinite (an infinite entry's have opposite signs, and entries of 2^104 and
// more, scaled, are) or a sum is.  A wave that has such outputs does its NB blocks of 16 x 16 from row m0 and output n0 on once more on the
// 32-bit unit and stores those outputs: `again` has the bit 4 t + e for output 4 g + e of block t.  (The whole wave comes here.)
template <int EPI, int NB>
__device__ __forceinline__ void redo(const Args& a, int m0, int n0, uint64_t again) {
  constexpr int SUMS = EPI == 1 ? 2 * NB : NB;
  if (__ballot(again != 0) == 0) return;
  const int lane = threadIdx.x % kWave, c = lane % 16, g = lane / 16;
  const float* const x = row_of(a.A, a.lda, m0 + c, a.M, g);
  const float* w[SUMS];
  floatx4 total[SUMS];
#pragma unroll
  for (int t = 0; t < SUMS; ++t) {
    w[t] = row_of(t < NB ? a.W : a.W2, a.K, n0 + t % NB * 16 + c, a.N, g);
    total[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  for (int k = 0; k < a.K; k += a.seg) plain_segment<SUMS>(x, w, k, a.K - k < a.seg ? a.K : k + a.seg, total);
  float* const out = a.C + static_cast<size_t>(m0 + c) * a.ldc + n0 + 4 * g;   // (lanes without a bit: not used)
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if ((again >> (4 * t + e)) & 1) out[t * 16 + e] = finish<EPI>(a, total[t][e], total[EPI == 1 ? NB + t : t][e]);
}

// blockDim: a wave per segment.  AROWS: rows of A that are read (8 or 16).
// PARTS: products of parts.  The rows' parts are made on the way into LDS (a lane's four columns), a weight's behind it.  Two
// stages ahead and two workgroups a CU (gated: 36 us for 47 with three and one, or four and one); for up to 8 rows of single
// weights four stages ahead, whose registers leave room for two workgroups too, and two stages' products side by side.
template <int EPI, int AROWS, bool PARTS>
__global__ __launch_bounds__(64 * kSegments, PARTS ? 4 : 1) void gemm_f32_few_kernel(Args a) {
  constexpr int NW = EPI == 1 ? 2 : 1, AP = AROWS / 8, D = PARTS && (EPI == 1 || AROWS == 16) ? 2 : 4;   // stages ahead
  constexpr int TOGETHER = PARTS && EPI != 1 && AROWS == 8 ? 2 : 1;   // stages whose products run side by side
  constexpr bool BUFFERS = TOGETHER == 2;
  constexpr int kAFloats = PARTS ? AROWS * BK * 3 / 2 : AROWS * BK;
  constexpr int kStageFloats = NW * 16 * BK + kAFloats, kWaveFloats = TOGETHER * kStageFloats;
  __shared__ __align__(16) float lds[kSegments * kWaveFloats];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int n0 = blockIdx.x * 16, r = lane / kPieces, p = lane % kPieces, c = lane % 16, g = lane / 16;
  const float sign = PARTS ? segment_sign(wave) : 1.f;
  const int k0 = wave * a.seg;
  const int k1 = a.K - k0 < a.seg ? a.K : k0 + a.seg;
  const int ns = (k1 - k0 + BK - 1) / BK;
  // Where a lane's rows begin.  BUFFERS (K < 4 Mi, rows less than 16 Mi apart): in bytes behind what all lanes share, for loads that add
  // the stage's columns, a scalar, themselves, where the vector unit has enough to do (256,000 outputs of 4 rows 387 us for 450; with 9 to
  // 16 rows the other kind is the faster one, 26 us for 30 against (2,304, 9,216)).
  using Rows = std::conditional_t<BUFFERS, int, const float*>;
  Rows wp[NW][2], ap[AP];
  const int here = a.N - n0 < 16 ? a.N - n0 : 16;
  const size_t tile = static_cast<size_t>(n0) * a.K;
  auto buffer = [](const float* p, int rows, int64_t stride, int K) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, static_cast<int>(((rows - 1) * stride + K) * 4), 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t w_buffer = buffer(a.W + tile, BUFFERS ? here : 1, a.K, a.K), a_buffer = buffer(a.A, BUFFERS ? a.M : 1, a.lda, a.K);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int n = 8 * i + r < here ? 8 * i + r : here - 1;
    if constexpr (BUFFERS) {
      wp[0][i] = (n * a.K + p * 4) * 4;
    } else {
      wp[0][i] = a.W + tile + static_cast<size_t>(n) * a.K;
      if (NW == 2) wp[NW - 1][i] = a.W2 + tile + static_cast<size_t>(n) * a.K;
    }
  }
#pragma unroll
  for (int i = 0; i < AP; ++i) {
    const int m = 8 * i + r < a.M ? 8 * i + r : a.M - 1;
    if constexpr (BUFFERS) ap[i] = (m * static_cast<int>(a.lda) + p * 4) * 4;
    else ap[i] = a.A + static_cast<size_t>(m) * a.lda;
  }
  floatx4 wv[D][NW][2], av[D][AP];
  auto load = [&](floatx4 (&w)[NW][2], floatx4 (&x)[AP], int s) __attribute__((always_inline)) {
    // (behind the segment's last stage: that one again; columns behind its end: its first ones, replaced by zeros below)
    const int at = k0 + (s < ns ? s : ns - 1) * BK;
    if constexpr (BUFFERS) {
#pragma unroll
      for (int i = 0; i < 2; ++i) w[0][i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(w_buffer, wp[0][i], at * 4, 0));
#pragma unroll
      for (int i = 0; i < AP; ++i) x[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(a_buffer, ap[i], at * 4, 0));
    } else {
      const int k = PARTS || at + p * 4 < k1 ? at + p * 4 : k0;
#pragma unroll
      for (int v = 0; v < NW; ++v)
#pragma unroll
        for (int i = 0; i < 2; ++i) w[v][i] = *reinterpret_cast<const floatx4*>(wp[v][i] + k);
#pragma unroll
      for (int i = 0; i < AP; ++i) x[i] = *reinterpret_cast<const floatx4*>(ap[i] + k);
    }
  };
  floatx4 acc[NW];
#pragma unroll
  for (int v = 0; v < NW; ++v) acc[v] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto to_lds = [&](const floatx4 (&w)[NW][2], const floatx4 (&x)[AP], int s, int area) __attribute__((always_inline)) {
    float* w_s = lds + wave * kWaveFloats + area * kStageFloats;
    float* a_s = w_s + NW * 16 * BK;
    const bool ok = PARTS || k0 + s * BK + p * 4 < k1;   // (products of parts: whole stages)
    const floatx4 zero{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < NW; ++v)
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<floatx4*>(w_s + v * 16 * BK + piece_at(8 * i + r, p)) = ok ? w[v][i] : zero;
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      if constexpr (PARTS) {   // a lane's four columns of a row, part by part: [part][column group][row][8]
        const float by = sign * kScale;
        float v[4] = {by * x[i][0], by * x[i][1], by * x[i][2], by * x[i][3]};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          typedef __attribute__((ext_vector_type(2))) uint32_t uint32x2;
          uint32x2 u;
          u[0] = round_two<true>(v[0], v[1]);
          u[1] = round_two<true>(v[2], v[3]);
          *reinterpret_cast<uint32x2*>(a_s + q * (AROWS * 16) + ((p % 4) * AROWS + 8 * i + r) * 4 + p / 4 * 2) = u;
        }
      } else {
        *reinterpret_cast<floatx4*>(a_s + piece_at(8 * i + r, p)) = ok ? x[i] : zero;
      }
    }
  };
  auto own_lds = [&]() __attribute__((always_inline)) {   // a wave's LDS accesses are carried out in their order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto multiply = [&](int area) __attribute__((always_inline)) {
    const float* w_s = lds + wave * kWaveFloats + area * kStageFloats;
    const float* a_s = w_s + NW * 16 * BK;
    if constexpr (PARTS) {
      Parts x;
#pragma unroll
      for (int q = 0; q < 3; ++q) x.p[q] = *reinterpret_cast<const bf16x8*>(a_s + q * (AROWS * 16) + (g * AROWS + c % AROWS) * 4);
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        const Parts w = parts<true>(kScale * *reinterpret_cast<const floatx4*>(w_s + v * 16 * BK + piece_at(c, g)),
                                    kScale * *reinterpret_cast<const floatx4*>(w_s + v * 16 * BK + piece_at(c, 4 + g)));
#pragma unroll
        for (int q = 0; q < kProducts; ++q)
          acc[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p[kPartOfW[q]], x.p[kPartOfX[q]], acc[v], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int b = 0; b < BK / 16; ++b) {
        const floatx4 x = *reinterpret_cast<const floatx4*>(a_s + piece_at(c % AROWS, b * 4 + g));
#pragma unroll
        for (int v = 0; v < NW; ++v) {
          const floatx4 w = *reinterpret_cast<const floatx4*>(w_s + v * 16 * BK + piece_at(c, b * 4 + g));
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], acc[v], 0, 0, 0);
        }
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(wv[d], av[d], d);
  int s = 0;
  for (; s + D <= ns; s += D) {
#pragma unroll
    for (int d = 0; d < D; d += TOGETHER) {
#pragma unroll
      for (int e = d; e < d + TOGETHER; ++e) to_lds(wv[e], av[e], s + e, e - d);
      own_lds();
#pragma unroll
      for (int e = d; e < d + TOGETHER; ++e) load(wv[e], av[e], s + e + D);
#pragma unroll
      for (int e = d; e < d + TOGETHER; ++e) multiply(e - d);
      own_lds();
    }
  }
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (s + d < ns) {   // (uniform over the wave; the loads are there)
      to_lds(wv[d], av[d], s + d, 0);
      own_lds();
      multiply(0);
      own_lds();
    }
  __syncthreads();
  floatx4* sums = reinterpret_cast<floatx4*>(lds);
  int* const infinite = reinterpret_cast<int*>(sums + kSegments * NW * kWave);   // of each segment: whether some sum of it is no finite number
  const int nseg = blockDim.x / kWave;
  auto put = [&](const floatx4 (&t)[NW]) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < NW; ++v) sums[(wave * NW + v) * kWave + lane] = t[v];
  };
  auto added = [&](floatx4 (&t)[NW]) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < NW; ++v) t[v] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < nseg; ++z)
#pragma unroll
      for (int v = 0; v < NW; ++v) t[v] += sums[(z * NW + v) * kWave + lane];
  };
  if constexpr (PARTS) {
    bool all = true;
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      acc[v] = sign * kUnscale * acc[v];
#pragma unroll
      for (int i = 0; i < 4; ++i) all = all && finite(acc[v][i]);
    }
    const bool some = __ballot(!all) != 0;
    if (lane == 0) infinite[wave] = some;
  }
  put(acc);
  __syncthreads();
  const bool stores = wave == 0 && c < a.M && n0 + 4 * g < a.N;
  floatx4 t[NW], y;
  int again = 0;
  if (wave == 0) {
    added(t);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[i] = finish<EPI>(a, t[0][i], t[NW - 1][i]);
      if (!(finite(t[0][i]) && finite(t[NW - 1][i]))) again |= 1 << i;
    }
    if (stores) store4(a, c, n0 + 4 * g, y);
  }
  if constexpr (PARTS) {   // (see redo; here a wave has its segment)
    int some = 0;
    for (int z = 0; z < nseg; ++z) some |= infinite[z];
    if (some == 0) return;
    int at = tid;
    asm("" : "+v"(at));
    const int cc = at % 16, gg = at % kWave / 16;
    const float* const x = row_of(a.A, a.lda, cc, a.M, gg);
    const float* w[NW];
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      w[v] = row_of(v == 0 ? a.W : a.W2, a.K, n0 + cc, a.N, gg);
      t[v] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    plain_segment<NW>(x, w, k0, k1, t);
    __syncthreads();   // (the sums of parts have been read)
    put(t);
    __syncthreads();
    if (!stores) return;
    added(t);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (((again >> i) & 1) && n0 + 4 * g + i < a.N)
        a.C[static_cast<size_t>(c) * a.ldc + n0 + 4 * g + i] = finish<EPI>(a, t[0][i], t[NW - 1][i]);
  }
}

// Tiles for K that is no multiple of 16 (or rows longer than 16 MB).  TM: blocks of 16 rows and of 16 weight rows of a wave; four
// waves, two by two.  With the gated epilogue half of a wave's weight rows are the gate's and half the other factor's of the same
// outputs.  PLANES: this workgroup's segment alone, its sums to planes [segment][M][columns] (gated: all the gate's columns, then
// the other factor's).
template <int EPI, int TM, bool PLANES>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(Args a, float* __restrict__ planes) {
  constexpr int ROWS = 2 * TM * 16;                 // rows of A, and rows of W, of a tile
  constexpr int LOADS = ROWS * kPieces / 256;
  constexpr int COLS = EPI == 1 ? ROWS / 2 : ROWS;  // outputs across
  constexpr int WT = EPI == 1 ? TM / 2 : TM;        // blocks of outputs across of a wave
  __shared__ __align__(16) float a_s[2][ROWS * BK];
  __shared__ __align__(16) float w_s[2][ROWS * BK];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave % 2, wn = wave / 2, c = lane % 16, g = lane / 16;
  const int m0 = blockIdx.y * ROWS, n0 = blockIdx.x * COLS;
  const int k0 = PLANES ? blockIdx.z * a.seg : 0;
  const int k1 = PLANES && k0 + a.seg < a.K ? k0 + a.seg : a.K;
  const int ns = (k1 - k0 + BK - 1) / BK, per_segment = a.seg / 16;
  const int r = tid / kPieces, p = tid % kPieces;   // 32 rows at a time
  const float* ap[LOADS];
  const float* wp[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = i * 32 + r;
    const int m = m0 + row < a.M ? m0 + row : a.M - 1;
    ap[i] = a.A + static_cast<size_t>(m) * a.lda;
    int n = n0 + row;
    const float* w = a.W;
    if (EPI == 1) {   // of a wave's TM * 16 rows the first half belongs to the gate
      const int in_wave = row % (TM * 16);
      n = n0 + row / (TM * 16) * (WT * 16) + in_wave % (WT * 16);
      if (in_wave >= WT * 16) w = a.W2;
    }
    wp[i] = w + static_cast<size_t>(n < a.N ? n : a.N - 1) * a.K;
  }
  floatx4 av[LOADS], wv[LOADS];
  auto load = [&](int s) __attribute__((always_inline)) {
    int k = k0 + (s < ns ? s : ns - 1) * BK + p * 4;
    k = k < k1 ? k : k0;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      av[i] = *reinterpret_cast<const floatx4*>(ap[i] + k);
      wv[i] = *reinterpret_cast<const floatx4*>(wp[i] + k);
    }
  };
  auto to_lds = [&](int s, int buf) __attribute__((always_inline)) {
    const bool ok = k0 + s * BK + p * 4 < k1;
    const floatx4 zero{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      *reinterpret_cast<floatx4*>(&a_s[buf][piece_at(i * 32 + r, p)]) = ok ? av[i] : zero;
      *reinterpret_cast<floatx4*>(&w_s[buf][piece_at(i * 32 + r, p)]) = ok ? wv[i] : zero;
    }
  };
  floatx4 acc[TM][TM], total[PLANES ? 1 : TM][TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (!PLANES) total[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  load(0);
  to_lds(0, 0);
  __syncthreads();
  int left = per_segment;
  for (int s = 0; s < ns; ++s) {
    const int buf = s & 1;
    load(s + 1);
#pragma unroll
    for (int b = 0; b < BK / 16; ++b) {
      floatx4 x[TM], w[TM];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        x[i] = *reinterpret_cast<const floatx4*>(&a_s[buf][piece_at((wm * TM + i) * 16 + c, b * 4 + g)]);
        w[i] = *reinterpret_cast<const floatx4*>(&w_s[buf][piece_at((wn * TM + i) * 16 + c, b * 4 + g)]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int t = 0; t < TM; ++t)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t][j], x[i][j], acc[i][t], 0, 0, 0);
      // a segment ends behind any block of 16; blocks behind K's end are zeros
      if (!PLANES && (--left == 0 || (s + 1 == ns && b + 1 == BK / 16))) {
        left = per_segment;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int t = 0; t < TM; ++t) {
            total[i][t] += acc[i][t];
            acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
    // (the other buffer's last readers passed the barrier of the stage before)
    if (s + 1 < ns) to_lds(s + 1, buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + c;
    if (m >= a.M) continue;
    if (PLANES) {
      const int64_t width = EPI == 1 ? 2 * static_cast<int64_t>(a.N) : a.N;
      Args b = a;
      b.C = planes + static_cast<size_t>(blockIdx.z) * a.M * width;
      b.ldc = width;
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        const int n = n0 + (wn * WT + t % WT) * 16 + 4 * g;
        Args to = b;
        if (EPI == 1 && t >= WT) to.C += a.N;
        if (n < a.N) store4(to, m, n, acc[i][t]);
      }
    } else {
#pragma unroll
      for (int t = 0; t < WT; ++t) {
        const int n = n0 + (wn * WT + t) * 16 + 4 * g;
        floatx4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = finish<EPI>(a, total[PLANES ? 0 : i][t][e], total[PLANES ? 0 : i][EPI == 1 ? t + WT : t][e]);
        if (n < a.N) store4(a, m, n, y);
      }
    }
  }
}

// Which tile: workgroups go to the eight XCDs in turn, each with an L2 of its own; an XCD gets a contiguous share of the tiles, and
// neighbours in it are up to eight tiles of rows against the same weights, which it reads from HBM once.
struct Tile {
  int x, y;
};
__device__ __forceinline__ Tile which_tile() {
  const int nx = gridDim.x, ny = gridDim.y, total = nx * ny;
  int l = blockIdx.x + nx * blockIdx.y;
  if (total % 8 == 0) l = (l % 8) * (total / 8) + l / 8;
  const int group = l / (8 * nx) * 8, height = ny - group < 8 ? ny - group : 8;
  l -= group * nx;
  return Tile{l / height, group + l % height};
}

// A load of 16 bytes a lane from global memory, `offset` bytes behind a base that all lanes share, straight into LDS: lane l's arrive
// at byte `lds` + 16 l.  The compiler does not know of it: arrived_barrier waits.
__device__ __forceinline__ void load_to_lds(const float* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(base), "s"(lds) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const float* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) float*)p));
}
// Every wave's loads into LDS have arrived but for its latest PENDING, and its reads of LDS are done.
template <int PENDING>
__device__ __forceinline__ void arrived_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(PENDING) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The same for K in multiples of 16, where nothing has to become zero on its way: loads go from global memory straight into LDS,
// and a wave's matrix instructions never wait for its operands.  TM x TN: blocks of 16 of a wave; WM x (4 / WM) waves.
// The fragments of a stage's two blocks of 16 columns have registers of their own; the products of the second block are held back
// behind the next barrier, where they cover the fragment reads of the next stage's first block, and the reads of the second are
// covered by the products of the first.  Reads and loads go out one by one, each behind some products: a wave issues in order,
// and more than the 32 cycles of one product between two of them leave the matrix unit idle (4,096 cubed: 117 TFLOP/s through
// registers, 125 with held-back products, 139.5 with the reads and loads spread; the unit's rate by itself is 155).
template <int EPI, int TM, int TN, int WM, int STAGES, bool PLANES>
__global__ __launch_bounds__(256, 2) void gemm_f32_flow_kernel(Args a, float* __restrict__ planes) {
  constexpr int WAVES = 4, WN = WAVES / WM, AR = WM * TM * 16, WR = WN * TN * 16;   // rows of A and of W of a tile
  constexpr int LA = AR / 8 / WAVES, LW = WR / 8 / WAVES, LOADS = LA + LW, PRODUCTS = 4 * TM * TN;
  constexpr int WT = EPI == 1 ? TN / 2 : TN;             // blocks of outputs across of a wave
  constexpr int STAGE = (AR + WR) * BK;
  static_assert(EPI != 1 || TN % 2 == 0, "half of a wave's weight rows are the gate's");
  __shared__ __align__(16) float stages[STAGES * STAGE];
  const uint32_t lds = lds_address(stages);
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave % WM, wn = wave / WM, c = lane % 16, g = lane / 16;
  const Tile tile = which_tile();
  const int m0 = tile.y * AR, n0 = tile.x * (WN * WT * 16);
  const int k0 = PLANES ? blockIdx.z * a.seg : 0;
  const int length = PLANES && k0 + a.seg < a.K ? a.seg : a.K - k0;   // a multiple of 16
  const int ns = (length + BK - 1) / BK, per_segment = a.seg / 16;
  // a load brings 8 rows of 128 bytes; lane l's piece arrives at 16 l, so the lane asks for the one that belongs there.  Of its
  // address the tile's and the stage's part are scalars, `off` is the rest, in bytes.
  const int r = lane / kPieces, at = ((lane % kPieces) ^ r) * 4;
  const float* const a_tile = a.A + static_cast<size_t>(m0) * a.lda + k0;
  const float* const w_tile = a.W + static_cast<size_t>(n0) * a.K + k0;
  const float* const w2_tile = EPI == 1 ? a.W2 + static_cast<size_t>(n0) * a.K + k0 : w_tile;
  uint32_t off[LOADS];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int m = (i * WAVES + wave) * 8 + r, last = a.M - 1 - m0;
    off[i] = (static_cast<uint32_t>(m < last ? m : last) * static_cast<uint32_t>(a.lda) + at) * 4;
  }
  // of a wave's TN * 16 weight rows the first half belongs to the gate (the 8 rows of a load are of one kind)
  auto of_gate = [&](int i) __attribute__((always_inline)) {
    return EPI != 1 || (i * WAVES + wave) * 8 % (TN * 16) < WT * 16;
  };
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    int n = (i * WAVES + wave) * 8 + r;
    const int last = a.N - 1 - n0;
    if (EPI == 1) n = n / (TN * 16) * (WT * 16) + n % (TN * 16) % (WT * 16);
    off[LA + i] = (static_cast<uint32_t>(n < last ? n : last) * static_cast<uint32_t>(a.K) + at) * 4;
  }
  // load i of stage s into a buffer (behind the last stage: that one again; columns behind the end: some of its own, not used)
  auto ask = [&](int i, int s, int buf) __attribute__((always_inline)) {
    const int k = (s < ns ? s : ns - 1) * BK;
    const uint32_t back = k + at < length ? 0u : 64u;
    const int row = i < LA ? i * WAVES * 8 : AR + (i - LA) * WAVES * 8;
    load_to_lds((i < LA ? a_tile : of_gate(i - LA) ? w_tile : w2_tile) + k, off[i] - back, lds + (buf * STAGE + (row + wave * 8) * BK) * 4);
  };
  floatx4 x[2][TM], w[2][TN];
  auto read = [&](int buf, int b, int i) __attribute__((always_inline)) {
    const float* stage = stages + buf * STAGE;
    if (i < TN) w[b][i] = *reinterpret_cast<const floatx4*>(stage + AR * BK + piece_at((wn * TN + i) * 16 + c, b * 4 + g));
    else x[b][i - TN] = *reinterpret_cast<const floatx4*>(stage + piece_at((wm * TM + i - TN) * 16 + c, b * 4 + g));
  };
  floatx4 acc[TM][TN], total[PLANES ? 1 : TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (!PLANES) total[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  auto end_of_segment = [&]() __attribute__((always_inline)) {
    if constexpr (!PLANES) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          total[i][t] += acc[i][t];
          acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  int left = per_segment;
  // The products of block b; meanwhile (next) block `to` of the stage in buffer `buf` is read, and (load) stage `stage` goes into
  // buffer `into`.
  auto multiply = [&](int b, bool next, int to, int buf, bool load, int stage, int into) __attribute__((always_inline)) {
    constexpr int READ_EVERY = PRODUCTS * 3 / 4 / (TM + TN), LOAD_EVERY = PRODUCTS / LOADS;
    static_assert(READ_EVERY >= 1 && LOAD_EVERY >= 1, "a product for each read and load");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b][t][j], x[b][i][j], acc[i][t], 0, 0, 0);
          const int q = (j * TM + i) * TN + t + 1;
          __builtin_amdgcn_sched_barrier(0);
          if (next && q % READ_EVERY == 0 && q / READ_EVERY <= TM + TN) read(buf, to, q / READ_EVERY - 1);
          if (load && q % LOAD_EVERY == 0 && q / LOAD_EVERY <= LOADS) ask(q / LOAD_EVERY - 1, stage, into);
          __builtin_amdgcn_sched_barrier(0);
        }
    if (!PLANES && --left == 0) {
      left = per_segment;
      end_of_segment();
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) ask(i, s, s);
  arrived_barrier<(STAGES - 1) * LOADS>();
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < TM + TN; ++i) read(0, b, i);
  multiply(0, false, 0, 0, false, 0, 0);
  int buf = 1, into = 0;
  for (int s = 1; s < ns; ++s) {
    arrived_barrier<(STAGES - 2) * LOADS>();   // everyone's loads of this stage; and everyone has read the stage before
    multiply(1, true, 0, buf, true, s + STAGES - 1, into);
    multiply(0, true, 1, buf, false, 0, 0);
    into = buf;
    buf = buf + 1 == STAGES ? 0 : buf + 1;
  }
  if (length % BK == 0) multiply(1, false, 0, 0, false, 0, 0);   // (uniform)
  if (!PLANES && left != per_segment) end_of_segment();
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");   // the loads asked for behind the last stage
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + c;
    if (m >= a.M) continue;
    if (PLANES) {
      const int64_t width = EPI == 1 ? 2 * static_cast<int64_t>(a.N) : a.N;
      Args b = a;
      b.C = planes + static_cast<size_t>(blockIdx.z) * a.M * width;
      b.ldc = width;
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const int n = n0 + (wn * WT + t % WT) * 16 + 4 * g;
        Args to = b;
        if (EPI == 1 && t >= WT) to.C += a.N;
        if (n < a.N) store4(to, m, n, acc[i][t]);
      }
    } else {
#pragma unroll
      for (int t = 0; t < WT; ++t) {
        const int n = n0 + (wn * WT + t) * 16 + 4 * g;
        floatx4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = finish<EPI>(a, total[PLANES ? 0 : i][t][e], total[PLANES ? 0 : i][EPI == 1 ? t + WT : t][e]);
        if (n < a.N) store4(a, m, n, y);
      }
    }
  }
}

// Where lane group g's eight numbers of a row lie in a part's KB (in bfloat16): neither the eight lanes that write together (two
// rows' four groups) nor the sixteen that read together (0-3, 12-15 and 20-27, and so on) meet in a bank.
__device__ __forceinline__ int part_at(int row, int g) {
  return (g * 16 + (row & 8) + ((g ^ (row / 2 % 4)) * 2) + row % 2) * 8;
}

// How a launch of products of parts goes over the tiles: the first `full` have a workgroup each, the others one for each segment.
struct Share {
  int nx, ny, full, nseg;
  float* planes;   // [tile - full][segment][block of 16 x 16 of a wave][thread] four sums
};
// The tile l of nx x ny: up to eight tiles of rows against the same weights are neighbours.
__device__ __forceinline__ Tile tile_at(const Share& s, int l) {
  const int group = l / (8 * s.nx) * 8, height = s.ny - group < 8 ? s.ny - group : 8;
  l -= group * s.nx;
  return Tile{l / height, group + l % height};
}

// Tiles of products of parts: eight waves, WM along the rows, TM x TN blocks of 16 a wave.  A workgroup makes the parts once, on
// their way from registers into LDS, in operand order: blocks of 16 rows x 32 columns, of each part 1 KB, in which lane 16 g + row
// reads its columns 4 g .. 4 g + 3 and 16 + 4 g .. (so that a load of 16 bytes by four lanes brings 64 neighbouring bytes).  Two
// buffers, one barrier a stage: a stage's products cover the next stage's parts, whose numbers were asked for a stage before.
template <int EPI, int TM, int TN, int WM, int WAVES>
__global__ __launch_bounds__(WAVES * kWave, 2) void gemm_f32_parts_kernel(Args a, Share share) {
  constexpr int THREADS = WAVES * kWave, WN = WAVES / WM, AB = WM * TM, WB = WN * TN;   // blocks of 16 rows of A and of W
  constexpr int BLOCKS = AB + WB, LOADS = (BLOCKS + WAVES - 1) / WAVES, BUF = BLOCKS * 3 * 512;
  // Gated: half of a wave's weight rows are the gate's; with an odd number of blocks a wave beside another has the gate's rows or the
  // other factor's, and the two exchange half of their sums at the end.  Such tiles' weight parts are read block by block.
  constexpr bool APART = TN % 2 == 1 && TN > 4, GATE_APART = EPI == 1 && APART;
  constexpr int WT = EPI == 1 && !APART ? TN / 2 : TN;   // blocks of outputs across of a wave
  constexpr int AGAIN = APART ? 3 : WT;                  // of them done again at a time
  static_assert(EPI != 1 || TN % 2 == 0 || (APART && WN == 2 && TM == 2), "gate and factor in one wave, or in two beside each other");
  static_assert(AB % WAVES == 0 && WT % AGAIN == 0, "a wave's first blocks are A's");
  __shared__ __align__(16) __bf16 lds[2 * BUF];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave % WM, wn = wave / WM, c = lane % 16, g = lane / 16;
  // workgroups go to the eight XCDs in turn, each with an L2 of its own: an XCD gets a contiguous share of the whole tiles
  int l = blockIdx.x, segment = -1;
  if (l < share.full) {
    if (share.full % 8 == 0) l = l % 8 * (share.full / 8) + l / 8;
  } else {
    segment = (l - share.full) % share.nseg;
    l = share.full + (l - share.full) / share.nseg;
  }
  const Tile tile = tile_at(share, l);
  const int m0 = tile.y * AB * 16, n0 = tile.x * ((GATE_APART ? 1 : WN) * WT * 16);
  const int k0 = segment < 0 ? 0 : segment * a.seg;
  const int length = segment >= 0 && k0 + a.seg < a.K ? a.seg : a.K - k0;   // a multiple of 32
  const int ns = length / BK, per_segment = a.seg / BK;
  const int r = lane / 4, p = lane % 4;
  // a load's address: the tile's part is the same for all lanes, the rest is an offset in elements (32 bits: K < 4 Mi, 288 rows)
  const float* const a_tile = a.A + static_cast<size_t>(m0) * a.lda + k0;
  const float* const w_tile = a.W + static_cast<size_t>(n0) * a.K + k0;
  const float* const w2_tile = EPI == 1 ? a.W2 + static_cast<size_t>(n0) * a.K + k0 : w_tile;
  uint32_t from[LOADS];
  auto mine = [&](int i) __attribute__((always_inline)) { return BLOCKS % WAVES == 0 || i * WAVES + wave < BLOCKS; };
  auto of_gate = [&](int i) __attribute__((always_inline)) {   // (the rows of a block are of one kind)
    const int n = i * WAVES + wave - AB;
    return EPI != 1 || (GATE_APART ? n < TN : n % TN < WT);
  };
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int b = mine(i) ? i * WAVES + wave : 0;
    if (i < AB / WAVES) {
      const int m = b * 16 + r, last = a.M - 1 - m0;
      from[i] = static_cast<uint32_t>(m < last ? m : last) * static_cast<uint32_t>(a.lda) + p * 4;
    } else {
      int n = b - AB;
      if (GATE_APART) n %= TN;
      else if (EPI == 1) n = n / TN * WT + n % TN % WT;   // of a wave's TN blocks the first half is the gate's
      const int row = (n < 0 ? 0 : n) * 16 + r, last = a.N - 1 - n0;
      from[i] = static_cast<uint32_t>(row < last ? row : last) * static_cast<uint32_t>(a.K) + p * 4;
    }
  }
  // signs and scales of the segments being summed and being made parts of, and stages that are left of each
  const float first = segment_sign(segment < 0 ? 0 : segment);
  float summed = first * kUnscale, prepared = first * kScale;
  int left = per_segment, to_prepare = per_segment;
  floatx4 v[LOADS][2];
  auto load = [&](int i, int s) __attribute__((always_inline)) {   // (behind the last stage: that one again)
    const int k = (s < ns ? s : ns - 1) * BK;
    const float* at = (i < AB / WAVES ? a_tile : of_gate(i) ? w_tile : w2_tile) + k;
    v[i][0] = *reinterpret_cast<const floatx4*>(at + from[i]);
    v[i][1] = *reinterpret_cast<const floatx4*>(at + from[i] + 16);
  };
  auto to_lds = [&](int i, int buf) __attribute__((always_inline)) {
    const float by = i < AB / WAVES ? prepared : kScale;
    const Parts x = parts(by * v[i][0], by * v[i][1]);
#pragma unroll
    for (int q = 0; q < 3; ++q)
      *reinterpret_cast<bf16x8*>(lds + buf * BUF + ((i * WAVES + wave) * 3 + q) * 512 + part_at(r, p)) = x.p[q];
  };
  auto read = [&](int buf, int b, int q) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8*>(lds + buf * BUF + (b * 3 + q) * 512 + part_at(c, g));
  };
  floatx4 acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[i][t] = total[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto end_of_segment = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        total[i][t] += summed * acc[i][t];
        acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
    left = per_segment, summed = -summed;
  };
  auto end_of_preparing = [&]() __attribute__((always_inline)) {
    if (--to_prepare == 0) to_prepare = per_segment, prepared = -prepared;
  };
  auto stage = [&](int s, int buf) __attribute__((always_inline)) {
    // this stage's parts are there and the other buffer's have been read; loads into registers stay under way
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (APART) {
      bf16x8 w[2][3], x[TM][3];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < 3; ++q) x[i][q] = read(buf, wm * TM + i, q);
#pragma unroll
      for (int q = 0; q < 3; ++q) w[0][q] = read(buf, AB + wn * TN, q);
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        if (t + 1 < TN) {
#pragma unroll
          for (int q = 0; q < 3; ++q) w[(t + 1) & 1][q] = read(buf, AB + wn * TN + t + 1, q);
        }
#pragma unroll
        for (int j = t * LOADS / TN; j < (t + 1) * LOADS / TN; ++j)
          if (mine(j)) {
            to_lds(j, buf ^ 1);
            load(j, s + 2);
          }
#pragma unroll
        for (int q = 0; q < kProducts; ++q)
#pragma unroll
          for (int i = 0; i < TM; ++i)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t & 1][kPartOfW[q]], x[i][kPartOfX[q]], acc[i][t], 0, 0, 0);
      }
    } else {
      bf16x8 w[TN][3], x[2][3];
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int q = 0; q < 3; ++q) w[t][q] = read(buf, AB + wn * TN + t, q);
#pragma unroll
      for (int q = 0; q < 3; ++q) x[0][q] = read(buf, wm * TM, q);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i + 1 < TM) {
#pragma unroll
          for (int q = 0; q < 3; ++q) x[(i + 1) & 1][q] = read(buf, wm * TM + i + 1, q);
        }
#pragma unroll
        for (int j = i * LOADS / TM; j < (i + 1) * LOADS / TM; ++j)
          if (mine(j)) {
            to_lds(j, buf ^ 1);
            load(j, s + 2);
          }
#pragma unroll
        for (int q = 0; q < kProducts; ++q)
#pragma unroll
          for (int t = 0; t < TN; ++t)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][kPartOfW[q]], x[i & 1][kPartOfX[q]], acc[i][t], 0, 0, 0);
      }
    }
    end_of_preparing();
    if (--left == 0) end_of_segment();
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    if (mine(i)) load(i, 0);
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    if (mine(i)) {
      to_lds(i, 0);
      load(i, 1);
    }
  end_of_preparing();
  int s = 0;
  for (; s + 1 < ns; s += 2) {
    stage(s, 0);
    stage(s + 1, 1);
  }
  if (s < ns) stage(s, 0);
  if (left != per_segment) end_of_segment();   // (a last segment that is shorter)
  if (segment >= 0) {
    floatx4* to = reinterpret_cast<floatx4*>(share.planes) +
                  (static_cast<size_t>(l - share.full) * share.nseg + segment) * (TM * TN * THREADS) + tid;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int t = 0; t < TN; ++t) to[(i * TN + t) * THREADS] = total[i][t];
    return;
  }
  if constexpr (GATE_APART) {   // the gate's wave keeps the first block of rows and gets the factor's sums of it, the other the second
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");   // the last stage's parts have been read
    floatx4* sums = reinterpret_cast<floatx4*>(lds);
#pragma unroll
    for (int t = 0; t < TN; ++t) sums[(wave * TN + t) * kWave + lane] = wn ? total[0][t] : total[1][t];
    __syncthreads();
    const int m = m0 + (wm * TM + wn) * 16 + c;
    uint64_t again = 0;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const int n = n0 + t * 16 + 4 * g;
      const floatx4 other = sums[((wm + WM * (1 - wn)) * TN + t) * kWave + lane];
      const floatx4 x = wn ? other : total[0][t], y = wn ? total[1][t] : other;
      floatx4 z;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (m < a.M && n + e < a.N && !(finite(x[e]) && finite(y[e]))) again |= 1ull << (t * 4 + e);
        z[e] = finish<EPI>(a, x[e], y[e]);
      }
      if (m < a.M && n < a.N) store4(a, m, n, z);
    }
    for (int t = 0; t < TN; t += AGAIN) redo<EPI, AGAIN>(a, m0 + (wm * TM + wn) * 16, n0 + t * 16, again >> (4 * t) & ((1ull << (4 * AGAIN)) - 1));
    return;
  }
  uint64_t again[TM];   // outputs whose sums are not finite: WT x 4 bits
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + c;
    again[i] = 0;
    if (m >= a.M) continue;
#pragma unroll
    for (int t = 0; t < WT; ++t) {
      const int n = n0 + (wn * WT + t) * 16 + 4 * g;
      floatx4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v0 = total[i][t][e], v1 = total[i][EPI == 1 && !APART ? t + WT : t][e];
        if (n + e < a.N && !(finite(v0) && finite(v1))) again[i] |= 1ull << (t * 4 + e);
        y[e] = finish<EPI>(a, v0, v1);
      }
      if (n < a.N) store4(a, m, n, y);
    }
  }
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {
    uint64_t of_row = 0;
#pragma unroll
    for (int j = 0; j < TM; ++j) of_row = j == i ? again[j] : of_row;
    for (int t = 0; t < WT; t += AGAIN)
      redo<EPI, AGAIN>(a, m0 + (wm * TM + i) * 16, n0 + (wn * WT + t) * 16, of_row >> (4 * t) & ((1ull << (4 * AGAIN)) - 1));
  }
}

// The tiles whose segments went to workgroups of their own: the segments' sums added in order.  gridDim: (blocks of outputs of a
// wave, tiles).
template <int EPI, int TM, int TN, int WM, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void gemm_f32_parts_sum_kernel(Args a, Share share) {
  constexpr int THREADS = WAVES * kWave, WN = WAVES / WM, WT = EPI == 1 ? TN / 2 : TN;
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave % WM, wn = wave / WM, c = lane % 16, g = lane / 16;
  const int i = blockIdx.x / WT, t = blockIdx.x % WT;
  const Tile tile = tile_at(share, share.full + blockIdx.y);
  const int m = tile.y * (WM * TM * 16) + (wm * TM + i) * 16 + c, n = tile.x * (WN * WT * 16) + (wn * WT + t) * 16 + 4 * g;
  const bool stores = m < a.M && n < a.N;
  if (__ballot(stores) == 0) return;   // (17 rows gated against (1,570, 256): 10.0 us for 11.6 with the planes of such waves read)
  const floatx4* from = reinterpret_cast<const floatx4*>(share.planes) +
                        (static_cast<size_t>(blockIdx.y) * share.nseg * (TM * TN) + i * TN + t) * THREADS + tid;
  floatx4 v[kSegments][EPI == 1 ? 2 : 1];
#pragma unroll
  for (int z = 0; z < kSegments; ++z) {   // (planes behind the last: the last again, not added)
    const floatx4* plane = from + static_cast<size_t>(z < share.nseg ? z : share.nseg - 1) * (TM * TN * THREADS);
    v[z][0] = plane[0];
    if constexpr (EPI == 1) v[z][1] = plane[WT * THREADS];
  }
  floatx4 x{0.f, 0.f, 0.f, 0.f}, y{0.f, 0.f, 0.f, 0.f}, to;
#pragma unroll
  for (int z = 0; z < kSegments; ++z)
    if (z < share.nseg) {
      x += v[z][0];
      if constexpr (EPI == 1) y += v[z][1];
    }
  uint64_t again = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (stores && n + e < a.N && !(finite(x[e]) && finite(y[e]))) again |= 1ull << e;
    to[e] = finish<EPI>(a, x[e], y[e]);
  }
  if (stores) store4(a, m, n, to);
  redo<EPI, 1>(a, m - c, n - 4 * g, again);
}

// C = epilogue(sum of the segments' planes, in order), V columns a thread.
template <int EPI, int V>
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(Args a, const float* __restrict__ planes, int nseg) {
  const size_t width = EPI == 1 ? 2 * static_cast<size_t>(a.N) : a.N, plane = static_cast<size_t>(a.M) * width;
  const size_t per_row = a.N / V, all = per_row * a.M;
  for (size_t e = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; e < all; e += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t m = e / per_row, n = e % per_row * V;
    const float* at = planes + m * width + n;
    float x[V], y[V];
#pragma unroll
    for (int i = 0; i < V; ++i) x[i] = y[i] = 0.f;
    float px[kSegments][V], py[EPI == 1 ? kSegments : 1][V];
#pragma unroll
    for (int z = 0; z < kSegments; ++z) {   // (planes behind the last: the last again, not added)
      const float* from = at + static_cast<size_t>(z < nseg ? z : nseg - 1) * plane;
      if constexpr (V == 4) {
        *reinterpret_cast<floatx4*>(px[z]) = *reinterpret_cast<const floatx4*>(from);
        if constexpr (EPI == 1) *reinterpret_cast<floatx4*>(py[z]) = *reinterpret_cast<const floatx4*>(from + a.N);
      } else {
        px[z][0] = from[0];
        if constexpr (EPI == 1) py[z][0] = from[a.N];
      }
    }
#pragma unroll
    for (int z = 0; z < kSegments; ++z)
#pragma unroll
      for (int i = 0; i < V; ++i) {
        if (z < nseg) x[i] += px[z][i];
        if constexpr (EPI == 1)
          if (z < nseg) y[i] += py[z][i];
      }
    float* dst = a.C + m * a.ldc + n;
    if constexpr (V == 4) {
      *reinterpret_cast<floatx4*>(dst) = floatx4{finish<EPI>(a, x[0], y[0]), finish<EPI>(a, x[1], y[1]),
                                                 finish<EPI>(a, x[2], y[2]), finish<EPI>(a, x[3], y[3])};
    } else {
      dst[0] = finish<EPI>(a, x[0], y[0]);
    }
  }
}

// Whether the products are gemm_f32_flow_kernel's: whole blocks of 16, and 128 rows' bytes in 32 bits.
static bool flows(int K, int64_t lda) { return K % 16 == 0 && K < (1 << 22) && lda < (1 << 22); }

struct Plan {
  int rows, cols;   // a tile's rows of A and of W; rows 16: few rows
  bool cut;         // products of parts: the tiles behind the last 256 whole ones
};

// Whether the products are those of parts: segments of whole stages (a matter of K alone but for rows of 64 MB and more apart, whose
// offsets in a tile take more than 32 bits).
static bool by_parts(int K, int seg, int64_t lda) { return K % BK == 0 && seg % BK == 0 && K < (1 << 22) && lda < (1 << 24); }

template <int EPI, bool PLANES>
static void launch_tile(const Args& a, const Plan& plan, int nseg, float* planes, hipStream_t stream) {
  const int cols = EPI == 1 ? plan.cols / 2 : plan.cols;
  const dim3 grid((a.N + cols - 1) / cols, (a.M + plan.rows - 1) / plan.rows, PLANES ? nseg : 1);
  if (!flows(a.K, a.lda)) {
    if (plan.rows == 128) gemm_f32_tile_kernel<EPI, 4, PLANES><<<grid, 256, 0, stream>>>(a, planes);
    else gemm_f32_tile_kernel<EPI, 2, PLANES><<<grid, 256, 0, stream>>>(a, planes);
    return;
  }
  if (plan.rows == 64) gemm_f32_flow_kernel<EPI, 2, 2, 2, 3, PLANES><<<grid, 256, 0, stream>>>(a, planes);
  else if (plan.cols == 64) gemm_f32_flow_kernel<EPI, 4, 2, 2, 2, PLANES><<<grid, 256, 0, stream>>>(a, planes);
  else if (plan.cols == 128) gemm_f32_flow_kernel<EPI, 4, 4, 2, 2, PLANES><<<grid, 256, 0, stream>>>(a, planes);
  else if constexpr (EPI == 1) gemm_f32_flow_kernel<EPI, 2, 6, 4, 2, PLANES><<<grid, 256, 0, stream>>>(a, planes);
  else gemm_f32_flow_kernel<EPI, 4, 3, 2, 2, PLANES><<<grid, 256, 0, stream>>>(a, planes);
}

template <int EPI, int TM, int TN, int WM, int WAVES>
static void launch_parts(const Args& a, const Plan& plan, int nseg, float* planes, hipStream_t stream) {
  constexpr int ROWS = WM * TM * 16, COLS = EPI == 1 ? WAVES / WM * TN * 8 : WAVES / WM * TN * 16, THREADS = WAVES * kWave;
  Share s;
  s.nx = (a.N + COLS - 1) / COLS, s.ny = (a.M + ROWS - 1) / ROWS, s.nseg = nseg, s.planes = planes;
  const int tiles = s.nx * s.ny;
  s.full = plan.cut ? tiles / 256 * 256 : tiles;
  gemm_f32_parts_kernel<EPI, TM, TN, WM, WAVES><<<s.full + (tiles - s.full) * nseg, THREADS, 0, stream>>>(a, s);
  if constexpr (EPI != 1 || TN % 2 == 0)
    if (s.full < tiles)
      gemm_f32_parts_sum_kernel<EPI, TM, TN, WM, WAVES><<<dim3(TM * (EPI == 1 ? TN / 2 : TN), tiles - s.full), THREADS, 0, stream>>>(a, s);
}

template <int EPI>
static void launch_tiles(const Args& a, const Plan& plan, int nseg, float* planes, hipStream_t stream) {
  if (planes == nullptr) {
    launch_tile<EPI, false>(a, plan, nseg, nullptr, stream);
    return;
  }
  launch_tile<EPI, true>(a, plan, nseg, planes, stream);
  const bool by_four = a.N % 4 == 0 && a.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(a.C) & 15u) == 0;
  const size_t all = static_cast<size_t>(a.M) * (a.N / (by_four ? 4 : 1));
  const int blocks = static_cast<int>((all + 255) / 256 > 4096 ? 4096 : (all + 255) / 256);
  if (by_four) gemm_f32_sum_kernel<EPI, 4><<<blocks, 256, 0, stream>>>(a, planes, nseg);
  else gemm_f32_sum_kernel<EPI, 1><<<blocks, 256, 0, stream>>>(a, planes, nseg);
}

// The tile and whether K is cut over workgroups: the workgroups that the busiest of 256 CUs gets, times a tile's products at the
// share of a CU's 614 GFLOP/s that the tile reaches, and for cut tiles the planes written and read at 4 TB/s and one launch more.
// The shares are what products of 512 rows and of 4,096 measured, with a start of 6 us; those of K that is no multiple of 16 the
// older kernel's.
static Plan plan_for(int M, int N, int K, int64_t lda, bool gated, int nseg, size_t workspace_bytes) {
  Plan best{16, 16, false};
  if (M <= 16) return best;
  struct Tile {
    int rows, cols;
    double share;
  };
  static const Tile flowing[4] = {{128, 128, 0.88}, {128, 96, 0.83}, {128, 64, 0.83}, {64, 64, 0.73}};
  static const Tile older[2] = {{128, 128, 0.85}, {64, 64, 0.7}};
  const bool flow = flows(K, lda);
  const double NW = gated ? 2.0 * N : N;
  const size_t plane_bytes = static_cast<size_t>(nseg) * M * static_cast<size_t>(NW) * sizeof(float);
  double best_us = 1e30;
  for (int i = 0; i < (flow ? 4 : 2); ++i) {
    const Tile& t = flow ? flowing[i] : older[i];
    const double tiles = ceil(M / static_cast<double>(t.rows)) * ceil(NW / t.cols);
    const double tile_us = 2.0 * t.rows * t.cols * K / (0.614e6 * t.share);
    for (int cut = 0; cut < 2; ++cut) {
      if (cut && (nseg == 1 || plane_bytes > workspace_bytes)) continue;
      const double us = cut ? ceil(tiles * nseg / 256.0) * tile_us / nseg + 2.0 * plane_bytes / 4e6 + 7.0
                            : ceil(tiles / 256.0) * tile_us + 6.0;
      if (us < best_us) best_us = us, best = Plan{t.rows, t.cols, cut != 0};
    }
  }
  return best;
}

// The same for products of parts: a round's start, its tiles at the rate that a CU reaches with them, the planes, the weights read
// once.  The figures of tiles of 64 x 128 and more are fitted to 4 to 11 ways of each of 61 to 1,024 rows against (9,216 gated, 2,304),
// (2,304, 9,216), (2,304, 2,048) and (4,096, 2,304), those of the small tiles to 17 to 4,096 rows against these and 39 other weights of
// 256 to 18,433 rows and K of 160 to 14,336.  128 x 288 is there for widths of whole such tiles where rounds of the others are half empty:
// 509 rows against (2,304, 9,216) 136 us for 152, against (2,304, 2,048) 40 for 47.  Gated ones are
// chosen for odd widths alone: at 24 such sizes, 1,300 to 2,048 rows of 2,064 to 3,283 outputs with K of 512 to 1,536, they are 0.98 to
// 1.19 times as fast as the best of the others, 1.09 in the mean (2,048 rows of 2,285 outputs, K = 512: 58 us for 70).
// Small tiles: of 64 x 64 for narrow weights (up to 3,072 rows), where larger ones leave CUs idle (17 rows against (1,024, 4,096) 16 us
// for 22, 1,024 against (512, 256) 9 for 17, 1,024 against (1,024, 1,024) 25 for 31) and for K up to 768 while they make two rounds at
// most (130 rows against (4,096, 512) 14 us for 20, (3,584, 736) 18 for 26, 100 against (1,570 gated, 256) 10.7 for 15.4), of 32 rows,
// cut, for what fills no more (17 rows against (9,216 gated, 2,304) 50 us for 59, (14,336 gated, 3,584) 98 for 118, (8,192, 3,584) 30
// for 37).  Over 436 sizes what is chosen takes 2 % more than the best way.  Not for up to 32 rows of wide weights with K of 256 and
// less, whose tiles are chosen as before, though smaller ones would be ahead (17 rows against (2,300 gated, 160): 8 us for 10).
static Plan plan_for_parts(int M, int N, int K, bool gated, int nseg, size_t workspace_bytes) {
  Plan best{16, 16, false};
  if (M <= 16) return best;
  struct Tile {
    int rows, cols, at_once;   // workgroups of a CU at a time
    double rate, start;        // FLOP a us of a CU, us
  };
  static const Tile tiles_of[9] = {{64, 128, 2, 0.65e6, 2.0}, {128, 64, 2, 0.66e6, 0.0}, {128, 128, 1, 0.84e6, 1.6}, {128, 192, 1, 0.98e6, 2.3},
                                   {128, 256, 1, 1.0e6, 1.9}, {128, 288, 1, 0.92e6, 1.6}, {64, 64, 3, 0.59e6, 0.5},  {32, 64, 4, 0.38e6, 0.15},
                                   {32, 128, 2, 0.38e6, 2.2}};
  const double NW = gated ? 2.0 * N : N;
  const bool narrow = NW <= 3072, one_stage = K <= kSegments * BK;   // (segments of one stage)
  const bool two_rounds = ceil(M / 64.0) * ceil(NW / 64.0) <= 512;   // of tiles of 64 x 64
  double best_us = 1e30;
  for (const Tile& t : tiles_of) {
    const bool rows_of_32 = t.rows == 32, of_64 = t.rows == 64 && t.cols == 64;
    if (gated && t.cols == 192) continue;   // (three blocks of a wave)
    if (rows_of_32 ? M > 32 || (one_stage && !narrow) || NW > 255.0 * t.cols : of_64 ? !narrow && !(M > 32 && K <= 768 && two_rounds) : narrow && one_stage && two_rounds) continue;
    const double tiles = ceil(M / static_cast<double>(t.rows)) * ceil(NW / t.cols), tile_us = 2.0 * t.rows * t.cols * K / t.rate;
    auto rounds = [&](double workgroups, double us) {
      const double of_a_cu = ceil(workgroups / 256.0);
      return of_a_cu * us + ceil(of_a_cu / t.at_once) * t.start;
    };
    for (int cut = rows_of_32; cut < 2; ++cut) {   // (whole, they have too little of the weights under way)
      const double rest = cut ? fmod(tiles, 256.0) : 0.0, plane_bytes = rest * nseg * t.rows * t.cols * sizeof(float);
      if (cut && (rest == 0 || nseg == 1 || plane_bytes > workspace_bytes || (gated && t.cols == 288))) continue;   // (no planes of those)
      if (one_stage && rest * nseg > 256.0) continue;   // (not worth a second workgroup of a CU: 509 rows against (512, 256) 8.7 us for 11)
      double us = rounds(tiles - rest, tile_us) + rounds(rest * nseg, tile_us / nseg) + 2.0 * plane_bytes / 7.9e6 + (cut ? 0.5 : 0.0);
      if (us < NW * K * sizeof(float) / 4.5e6) us = NW * K * sizeof(float) / 4.5e6;
      if (us < best_us) best_us = us, best = Plan{t.rows, t.cols, cut != 0};
    }
  }
  return best;
}

// Segments of K, and their length.
static int segments(int K, int* length) {
  *length = (K + kSegments * 16 - 1) / (kSegments * 16) * 16;
  return (K + *length - 1) / *length;
}

template <int EPI>
static void launch(const Args& a, int nseg, float* workspace, size_t workspace_bytes, hipStream_t stream) {
  const size_t planes_bytes = workspace != nullptr ? workspace_bytes : 0;
  const Plan plan = a.parts ? plan_for_parts(a.M, a.N, a.K, EPI == 1, nseg, planes_bytes)
                            : plan_for(a.M, a.N, a.K, a.lda, EPI == 1, nseg, planes_bytes);
  if (plan.rows == 16) {
    const int blocks = (a.N + 15) / 16;
    if (a.parts) {
      if (a.M <= 8) gemm_f32_few_kernel<EPI, 8, true><<<blocks, 64 * nseg, 0, stream>>>(a);
      else gemm_f32_few_kernel<EPI, 16, true><<<blocks, 64 * nseg, 0, stream>>>(a);
    } else if (a.M <= 8) {
      gemm_f32_few_kernel<EPI, 8, false><<<blocks, 64 * nseg, 0, stream>>>(a);
    } else {
      gemm_f32_few_kernel<EPI, 16, false><<<blocks, 64 * nseg, 0, stream>>>(a);
    }
    return;
  }
  if (a.parts) {
    if (plan.rows == 32 && plan.cols == 64) launch_parts<EPI, 2, 2, 1, 2>(a, plan, nseg, workspace, stream);
    else if (plan.rows == 32) launch_parts<EPI, 2, 4, 1, 2>(a, plan, nseg, workspace, stream);
    else if (plan.rows == 64 && plan.cols == 64) launch_parts<EPI, 2, 2, 2, 4>(a, plan, nseg, workspace, stream);
    else if (plan.rows == 64) launch_parts<EPI, 2, 4, 2, 4>(a, plan, nseg, workspace, stream);
    else if (plan.cols == 64) launch_parts<EPI, 4, 2, 2, 4>(a, plan, nseg, workspace, stream);
    else if (plan.cols == 128) launch_parts<EPI, 4, 2, 2, 8>(a, plan, nseg, workspace, stream);
    else if (plan.cols == 256) launch_parts<EPI, 4, 4, 2, 8>(a, plan, nseg, workspace, stream);
    else if (plan.cols == 288) launch_parts<EPI, 2, 9, 4, 8>(a, plan, nseg, workspace, stream);
    else if constexpr (EPI != 1) launch_parts<EPI, 4, 3, 2, 8>(a, plan, nseg, workspace, stream);
    return;
  }
  launch_tiles<EPI>(a, plan, nseg, plan.cut ? workspace : nullptr, stream);
}

}  // namespace f32

bool gemm_f32_takes(int M, int N, int K, int64_t lda, const void* A, const void* W, const void* W2) {
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  return M >= 1 && K % 4 == 0 && lda % 4 == 0 && aligned(A) && aligned(W) && aligned(W2) && N <= (1 << 30) / 16 &&
         (M + 63) / 64 <= 65535;   // (tiles of rows are the grid's second index)
}

int gemm_f32(const float* A, int64_t lda, const float* W, const float* W2, float* C, int64_t ldc, int M, int N, int K, int epi,
             int act, float cap, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  f32::Args a;
  a.A = A, a.W = W, a.W2 = W2, a.C = C, a.lda = lda, a.ldc = ldc, a.M = M, a.N = N, a.K = K, a.act = act, a.cap = cap;
  const int nseg = f32::segments(K, &a.seg);
  a.parts = f32::by_parts(K, a.seg, lda);
  float* ws = static_cast<float*>(workspace);
  if (epi == kEpilogueGated) f32::launch<1>(a, nseg, ws, workspace_bytes, stream);
  else if (epi == kEpilogueSoftCap) f32::launch<2>(a, nseg, ws, workspace_bytes, stream);
  else f32::launch<0>(a, nseg, ws, workspace_bytes, stream);
  return check_launch("gemm_f32");
}

}  // namespace sa

// Which way M rows go: 16 (few rows), or a tile's rows (64 or 128), plus 1000 where K is cut over workgroups, plus 10000 times the
// weight rows of a tile.
extern "C" int sa_gemm_f32_plan(int M, int N, int K, int gated, int64_t workspace_bytes) {
  if (M < 1 || N < 1 || K < 1) return 0;
  int length;
  const int nseg = sa::f32::segments(K, &length);
  const size_t bytes = workspace_bytes > 0 ? static_cast<size_t>(workspace_bytes) : 0;
  const sa::f32::Plan plan = sa::f32::by_parts(K, length, K) ? sa::f32::plan_for_parts(M, N, K, gated != 0, nseg, bytes)
                                                          : sa::f32::plan_for(M, N, K, K, gated != 0, nseg, bytes);
  return plan.rows + (plan.cut ? 1000 : 0) + 10000 * plan.cols;
}
