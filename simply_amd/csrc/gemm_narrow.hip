// C[M, N] = A[M, K] . W[N, K]^T in bfloat16 for many rows against at most 64 outputs (a router, gates, the first factor of a low-rank
// map): bound by the start of a launch and one read of the rows (8 MB at 2,048 rows of 2,048).
//
// A workgroup takes 16 rows and all outputs, its eight waves an eighth of K each.  A wave loads the rows' fragments (16 rows x 64
// bytes) and the weights' straight into registers, four columns of fragments at a time, and nothing goes through LDS but the
// eight waves' sums, which are added in the waves' order: a row's sums run the same way whatever rows are beside it.
// K a multiple of 32, W tiled.
//
// us in a graph of launches, 32-bit results, before (the tiled kernel, mostly with K cut and a sum kernel) / now, K = 2,048: 16 outputs 33
// rows 8.4 / 4.2, 774 9.9 / 4.3, 2,047 11 / 4.4, 8,192 20.5 / 7.2; 64 outputs 8.7 / 6.3, 11.8 / 6.5, 13.0 / 6.6, 22.2 / 12.0; K = 4,096, 64
// outputs, 33 rows 9.5 / 9.8, 2,047 16.1 / 10.6.  A CU's loads are what it then waits for: sixteen waves take as long (10.6 there), the
// loads left to the compiler's order, a few at a time, up to 9 % longer.  For 17 to 32 rows the few-rows kernel takes as long (16
// outputs 4.7 / 4.0, 64 4.9 / 5.7) and keeps them.
#include "api.h"
#include "common.h"

namespace sa {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

namespace narrow {

constexpr int kWaves = 8, kUnroll = 4;

template <int NT>
__global__ __launch_bounds__(kWaves * kWave) void gemm_narrow_kernel(const bf16* __restrict__ A, int64_t lda, const bf16* __restrict__ W,
                                                                  void* __restrict__ C, int c_dtype, int64_t ldc, int M, int N, int chunks) {
  __shared__ floatx4 sums[kWaves][NT][kWave];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c0 = chunks * wave / kWaves, c1 = chunks * (wave + 1) / kWaves;
  const int m0 = blockIdx.x * 16;
  const int row = m0 + lane % 16 < M ? m0 + lane % 16 : M - 1;   // (rows beyond the last are not stored)
  const bf16* a = A + row * lda + lane / 16 * 8;
  const bf16* w = W + lane * 8;
  const size_t tile = static_cast<size_t>(chunks) * 512;
  floatx4 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto several = [&](int c, auto count_tag) __attribute__((always_inline)) {
    constexpr int COUNT = decltype(count_tag)::value;
    bf16x8 fa[COUNT], fw[COUNT][NT];
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
      fa[u] = *reinterpret_cast<const bf16x8*>(a + (c + u) * 32);
#pragma unroll
      for (int j = 0; j < NT; ++j) fw[u][j] = *reinterpret_cast<const bf16x8*>(w + j * tile + static_cast<size_t>(c + u) * 512);
    }
    __builtin_amdgcn_sched_barrier(0);   // all of them under way before the first is waited for
#pragma unroll
    for (int u = 0; u < COUNT; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[u][j], fa[u], acc[j], 0, 0, 0);
  };
  int c = c0;
  for (; c + kUnroll <= c1; c += kUnroll) several(c, std::integral_constant<int, kUnroll>{});
  for (; c < c1; ++c) several(c, std::integral_constant<int, 1>{});
#pragma unroll
  for (int j = 0; j < NT; ++j) sums[wave][j][lane] = acc[j];
  __syncthreads();
  // lane l of tile j holds outputs 16 j + 4 (l / 16) .. of row l % 16
  for (int j = wave; j < NT; j += kWaves) {
    floatx4 total = sums[0][j][lane];
#pragma unroll
    for (int v = 1; v < kWaves; ++v) total += sums[v][j][lane];
    const int m = m0 + lane % 16, n = j * 16 + lane / 16 * 4;
    if (m >= M) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) store_f(C, c_dtype, static_cast<size_t>(m) * ldc + n + e, total[e]);
  }
}

}  // namespace narrow

// Microseconds of a launch among others: the loads of 16 rows and all weights by every CU, as many times as it gets 16 rows, or all rows
// once (within 14 % of the measured time of 8 to 64 outputs up to 2,047 rows of K = 512 to 36,864 and up to 8,192 of 4,096; beyond, where
// this kernel is far ahead, it takes up to 1.8 times as long).
static double narrow_us(int M, int N, int K) {
  const double times = fmax(1.0, (M + 15) / 16 / 256.0);
  return 2.1 + fmax(times * K / 1024.0 * (0.79 + 0.27 * ((N + 15) / 16)), static_cast<double>(M) * K * 2 / 6e6);
}

// Up to K = 4,096 always (which kernel a row meets does not depend on its neighbours there; the one size that loses is 33 rows against 64
// outputs, 9.5 / 9.8 us).  A longer K, of which a workgroup walks all by itself, is left to the tiled kernel with its cuts of K, whose time
// for so few outputs is the second figure, until there are rows for many workgroups; us, tiled / this, 32-bit results: K = 8,192, 16
// outputs 33 rows 10.2 / 10.8, 200 12.0 / 11.0, 64 outputs 200 13.5 / 17.3, 2,047 22 / 18; 16,384, 16 outputs 200 15 / 20, 1,031 23 / 20, 64
// outputs 1,031 24 / 32, 4,096 60 / 36; 36,864, 16 outputs 33 rows 19 / 41, 1,031 39 / 41, 2,047 64 / 42, 64 outputs 33 rows 21 / 70, 2,047
// 72 / 74, 4,096 158 / 115.
bool gemm_narrow_takes(int M, int N, int K) {
  return M > 32 && N <= 64 && K % 32 == 0 &&
         (K <= 4096 || narrow_us(M, N, K) <= 7.0 + 0.03 * (M < 64 ? M : 64) + 0.28 * K / 1024 + static_cast<double>(M) * K * 2 / 3.6e6);
}

// (the wide kernel's small tiles are 1 to 3 us below their figure at these sizes)
double gemm_narrow_predict_us(int M, int N, int K) { return 0.5 + narrow_us(M, N, K); }

int gemm_narrow(const void* A, int64_t lda, const void* W, void* C, int c_dtype, int64_t ldc, int M, int N, int K, hipStream_t stream) {
  const bf16* a = static_cast<const bf16*>(A);
  const bf16* w = static_cast<const bf16*>(W);
  const int groups = (M + 15) / 16, tiles = (N + 15) / 16;
#define SA_NARROW(NT) narrow::gemm_narrow_kernel<NT><<<groups, narrow::kWaves * kWave, 0, stream>>>(a, lda, w, C, c_dtype, ldc, M, N, K / 32)
  if (tiles <= 1) SA_NARROW(1);
  else if (tiles == 2) SA_NARROW(2);
  else if (tiles == 3) SA_NARROW(3);
  else SA_NARROW(4);
#undef SA_NARROW
  return check_launch("gemm_narrow");
}

}  // namespace sa

extern "C" int sa_gemm_narrow_takes(int M, int N, int K) { return M > 0 && N > 0 && K > 0 && sa::gemm_narrow_takes(M, N, K); }
