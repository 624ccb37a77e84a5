// C[M, N] = epilogue(A[M, K] . W[N, K]^T) in bfloat16 for many rows, on the largest tiles that a CU's registers hold: a workgroup of
// four waves, one to a SIMD, has 256 x 288, 256 x 256, 192 x 288 or 192 x 256 outputs, a wave a quarter of them.
//   * What bounds it: the matrix units' power.  With every CU at work they are busy 72 % of the cycles at 1.93 GHz (2,048 rows, 8,192
//     outputs, K = 8,192: 188 us, 1.46 PFLOP/s); with the loads left out the same loop takes 22 % less time, in part by the clock.
//     A wave's 128 x 144 outputs need 17 fragment reads for 72 products where the wide kernel's 64 x 96 need 10 for 24, and a tile of
//     256 x 288 brings 34 KiB into LDS for 72 products a SIMD where two of 128 x 192 bring 40 for 48: what is moved for a product
//     is what power can be saved on.
//   * Layout in LDS: W as KiB blocks in MFMA operand order, which is how it lies in global memory, in a ring of halves (32 columns
//     of K); A as rows of 128 bytes (whole lines), their 16-byte pieces permuted by the row's number against bank conflicts, in a
//     ring of slabs (64 columns).  The rings are as deep as 160 KiB allow: three slabs of A, three or four halves of W, so that a
//     load has the time of two halves and more (1.2 us and more) for its way from HBM.
//   * Schedule of a half: one barrier; then its products, with the fragments of the next half read one by one between the first of
//     them into registers of their own, and this half's share of the loads spread over all of them.  A wave waits for nothing in between.
//   * The products are instructions written out ("+a": a sum stays in its registers).  Left to the compiler's intrinsic, 16 to 200
//     copies of sums a slab stood in the loop, each a wait for the matrix unit: 88 us for 2,048 x 8,192 x 2,048, now 54 to 57.
//   * The results go through LDS as bfloat16: whole rows are stored, and an activation's code stands in the kernel once for each rule
//     (unrolled over a wave's registers it was 100 KiB of code, 13 us of cold instruction fetches a launch).
// Before (the wide kernel) and now, us: gated, 2,048 rows of the 2B feed-forward 159 / 134, 8,192 rows 578 / 511, 1,056
// rows of the 27B one 649 / 593; 2,048 rows against 8,192 outputs of K = 2,048 66 / 56, 4,096 cubed 110 / 95.
#include "api.h"
#include "slabs.h"

namespace sa {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

namespace broad {

using slabs::bare_barrier;
using slabs::waitcnt_vm;

constexpr int BK = 64;      // columns of K of a slab of A; W goes by halves of 32
constexpr int kCUs = 256;

template <int N> struct Int { static constexpr int value = N; };
template <int N, int AT = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (AT < N) {
    f(Int<AT>{});
    each<N, AT + 1>(f);
  }
}

// Two values rounded to bfloat16, the first in the lower half: one instruction (one by one they take a shift and an or besides).
__device__ __forceinline__ uint32_t two_bf16(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float floatx2;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{a, b}), bf16x2));
}

// 16 bytes per lane from base + offset + FROM bytes into LDS at byte address lds + TO + 16 * lane
template <int FROM, int TO>
__device__ __forceinline__ void load_block(const bf16* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3"
               :
               : "v"(offset), "s"(base), "s"(lds), "n"(FROM), "n"(TO)
               : "memory", "scc");
}

// WM x WN: 16 x 16 tiles of a wave (rows of A x rows of W); RA slabs of A and RW halves of W in LDS.  EPI 0: none, or (act > 0) the
// activation act - 1 of the product rounded to bfloat16; 1: gated (tiles of W alternate between the two factors); 3: the 32-bit
// sums of this workgroup's share of K (gridDim.z of them) to `partials` [z][M][N].
template <int WM, int WN, int RA, int RW, int EPI>
__global__ __launch_bounds__(256, 1) void gemm_broad_kernel(const bf16* __restrict__ A, int64_t lda,
                                                         const bf16* __restrict__ W, bf16* __restrict__ C, int64_t ldc,
                                                         int M, int N, int K, int chunks, int act, float limit,
                                                         float* __restrict__ partials, Sections sec) {
  constexpr int MT = 2 * WM, NT = 2 * WN;
  constexpr int BM = MT * 16;
  constexpr int A_SLAB = MT * 1024, W_HALF = NT * 512;         // elements
  constexpr int LA = MT / 4, LW = (NT + 3) / 4;                // loads of a wave in a half
  constexpr int GROUP = LA + LW;
  constexpr int WNE = WN & ~1;
  static_assert(MT % 4 == 0, "every wave copies the same number of blocks of A");
  __shared__ __attribute__((aligned(16))) __bf16 lds[RA * A_SLAB + RW * W_HALF];
  const uint32_t lds_a = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) __bf16*)lds));

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / 2, wn = wave % 2;
  // Which tile: as in the wide kernel, an XCD gets a contiguous share of the tiles, in columns eight wide, rows first.
  int bx = blockIdx.x, by = blockIdx.y;
  {
    const int nx = gridDim.x, ny = gridDim.y, total = nx * ny;
    int l = bx + nx * by;
    if (total % 8 == 0) l = (l % 8) * (total / 8) + l / 8;
    constexpr int GX = 8;
    const int full = nx / GX;
    if (l < full * GX * ny) {
      const int col = l / (GX * ny), rem = l % (GX * ny);
      by = rem / GX;
      bx = col * GX + rem % GX;
    } else {
      const int rem = l - full * GX * ny, width = nx % GX;
      by = rem / width;
      bx = full * GX + rem % width;
    }
  }
  const int slabs_all = K / BK;
  const int slab0 = blockIdx.z * slabs_all / gridDim.z;
  const int slabs = (blockIdx.z + 1) * slabs_all / gridDim.z - slab0;
  const int m_base = by * BM;
  const int NW = EPI == 1 ? 2 * ((N + 15) / 16) * 16 : N;
  // several products at once: which section this workgroup is in, its columns of A, its rows of W
  int first_tile = 0, NL = NW;   // the section's first 16-row tile of W and the end of its rows
  if (EPI == 0 && sec.n_step > 0) {
    const int per = (sec.n_step + NT * 16 - 1) / (NT * 16), s = bx / per;
    bx -= s * per;
    first_tile = s * (sec.n_step / 16);
    A += static_cast<size_t>(s) * sec.a_step;
    NL = (s + 1) * sec.n_step < NW ? (s + 1) * sec.n_step : NW;
  }
  const int ntiles = (NL + 15) / 16;
  const int nt_base = first_tile + bx * NT;

  // ---- what this wave copies: of a slab of A the KiB blocks (tile tile_mine + 2 i, its rows 8 half_mine ..), half of them in each
  // half; of a half of W the tiles wave + 4 i.  Rows beyond M read row M - 1, tiles beyond the last the last one (never stored).
  const int half_mine = wave % 2, tile_mine = wave / 2;
  uint32_t a_off[2 * LA], w_off[LW];
#pragma unroll
  for (int i = 0; i < 2 * LA; ++i) {
    const int r = half_mine * 8 + lane / 8;
    const int m = m_base + (tile_mine + 2 * i) * 16 + r;
    const int from = m < M ? m : M - 1;
    a_off[i] = (static_cast<uint32_t>(from) * static_cast<uint32_t>(lda) + ((lane % 8) ^ (r / 2)) * 8) * 2;
  }
  // block i of a half: tile wave + 4 i (a wave that has no such tile loads its block before once more)
  auto w_tile = [&](int i) { return wave + 4 * i < NT ? wave + 4 * i : wave + 4 * (i - 1); };
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int nt = nt_base + w_tile(i);
    w_off[i] = static_cast<uint32_t>((nt < ntiles ? nt : ntiles - 1) - nt_base) * chunks * 1024 + lane * 16;
  }
  A += static_cast<size_t>(slab0) * BK;
  W += (static_cast<size_t>(nt_base) * chunks + static_cast<size_t>(slab0) * 2) * 512;
  const uint32_t a_to_mine = lds_a + (tile_mine * 2 + half_mine) * 1024;
  const uint32_t w_to_mine = lds_a + RA * A_SLAB * 2 + wave * 1024, w_to_last = lds_a + RA * A_SLAB * 2 + w_tile(LW - 1) * 1024;
  // (past the last slab the last one is loaded again: no branch, and nothing is read beyond the operands)
  auto a_slab_at = [&](int slab) { return A + static_cast<size_t>(slab < slabs ? slab : slabs - 1) * BK; };
  auto w_half_at = [&](int half) { return W + static_cast<size_t>(half < 2 * slabs ? half : 2 * slabs - 1) * 512; };
  auto request_w = [&](auto n_tag, const bf16* at, int slot) __attribute__((always_inline)) {
    constexpr int n = decltype(n_tag)::value;
    if constexpr (4 * n + 4 <= NT) load_block<0, 4 * n * 1024>(at, w_off[n], w_to_mine + slot * (W_HALF * 2));
    else load_block<0, 0>(at, w_off[n], w_to_last + slot * (W_HALF * 2));
  };
  auto request_a = [&](auto i_tag, const bf16* at, int slot) __attribute__((always_inline)) {
    constexpr int i = decltype(i_tag)::value;
    load_block<0, i * 4096>(at, a_off[i], a_to_mine + slot * (A_SLAB * 2));
  };

  floatx4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  // The products are instructions written out, so that every sum keeps its registers (the compiler's own choice of them moves
  // dozens of sums around in every slab).  It inserts no waits between such a product and what it does with the sums itself:
  // here they are, and all that it does with them comes before or after.
  constexpr int IN_A = 64;   // sums in accumulation registers; the others in vector registers
  auto settle = [&]() __attribute__((always_inline)) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    each<WM * WN>([&](auto q_tag) __attribute__((always_inline)) {
      constexpr int q = decltype(q_tag)::value;
      floatx4& sum = acc[q / WN][q % WN];
      if constexpr (q < IN_A) asm volatile("" : "+a"(sum));
      else asm volatile("" : "+v"(sum));
    });
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  };
  settle();
  int a_frag[2];
#pragma unroll
  for (int kc = 0; kc < 2; ++kc) {
    const int r = lane % 16;
    a_frag[kc] = wm * WM * 1024 + r * 64 + ((kc * 4 + lane / 16) ^ (r / 2)) * 8;
  }
  // the 16-row tiles of W of a wave: WNE neighbours, and of an odd number one of the last two
  const int w_frag = (wn * WNE * 64 + lane) * 8, w_frag_last = ((2 * WNE + wn) * 64 + lane) * 8;
  auto tile_of = [&](int j) { return j < WNE ? wn * WNE + j : 2 * WNE + wn; };
  bf16x8 fa[2][WM], fw[2][WN];
  auto read_one = [&](auto set_tag, auto n_tag, int a_slot, int w_slot) __attribute__((always_inline)) {
    constexpr int set = decltype(set_tag)::value, n = decltype(n_tag)::value;
    if constexpr (n < WNE) fw[set][n] = *reinterpret_cast<const bf16x8*>(lds + RA * A_SLAB + w_slot * W_HALF + w_frag + n * 512);
    else if constexpr (n < WN) fw[set][n] = *reinterpret_cast<const bf16x8*>(lds + RA * A_SLAB + w_slot * W_HALF + w_frag_last);
    else fa[set][n - WN] = *reinterpret_cast<const bf16x8*>(lds + a_slot * A_SLAB + (n - WN) * 1024 + a_frag[set]);
  };

  // ---- The loads go in groups, one a half.  Group h, asked for after the barrier of half h: half h + RW of W, into the place of half
  // h, and of A half a slab: in the second half of slab t the first part of slab t + RA, into the place of slab t, in the half after
  // it the second part.  (The places are free: their fragments were read in the half before, and the barrier has been since.)
  // At the barrier of half h there must be what the reads in it want, half h + 1: loads of group h - AHEAD and before.
  // Before the loop: the groups of the halves before the first.
  constexpr int AHEAD_W = RW - 1, AHEAD_A = 2 * RA - 3, AHEAD = AHEAD_W < AHEAD_A ? AHEAD_W : AHEAD_A;
  constexpr int BEHIND = (AHEAD - 1) * GROUP + (AHEAD_W < AHEAD_A ? LA : 0);   // loads that may be under way at a half's barrier
  constexpr int BEFORE = RW > 2 * RA - 1 ? RW : 2 * RA - 1;
  static_assert(BEFORE * GROUP < 64, "loads under way are counted in six bits");
  each<BEFORE>([&](auto tag) __attribute__((always_inline)) {
    constexpr int g = decltype(tag)::value - BEFORE, w_half = g + RW, part = g % 2 == 0 ? 1 : 0;
    constexpr int a_slab = (g - 1 - part + 2 * RA) / 2;
    if constexpr (w_half >= 0)
      each<LW>([&](auto n) __attribute__((always_inline)) { request_w(n, w_half_at(w_half), w_half); });
    if constexpr (g >= 1 - 2 * RA)
      each<LA>([&](auto n) __attribute__((always_inline)) { request_a(Int<part * LA + decltype(n)::value>{}, a_slab_at(a_slab), a_slab); });
  });
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(BEHIND + GROUP));
  bare_barrier();
  each<WM + WN>([&](auto n) __attribute__((always_inline)) { read_one(Int<0>{}, n, 0, 0); });

  // one half: products of set SET, reads for the next half, loads of the half's group
  auto half_step = [&](auto set_tag, int a_next, int w_next, const bf16* w_at, int w_slot, const bf16* a_at, int a_slot)
                       __attribute__((always_inline)) {
    constexpr int SET = decltype(set_tag)::value, P = WM * WN, LOAD_EVERY = P / GROUP;
    constexpr int READ_EVERY = P / (WM + WN) < 3 ? P / (WM + WN) : 3;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(BEHIND) & ~(15 << 8));
    bare_barrier();
    each<P>([&](auto q_tag) __attribute__((always_inline)) {
      constexpr int q = decltype(q_tag)::value, i = q / WN, j = q % WN;
      if constexpr (q < IN_A) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fw[SET][j]), "v"(fa[SET][i]));
      else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(fw[SET][j]), "v"(fa[SET][i]));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (q % READ_EVERY == 0 && q / READ_EVERY < WM + WN) read_one(Int<1 - SET>{}, Int<q / READ_EVERY>{}, a_next, w_next);
      if constexpr (q % LOAD_EVERY == 1 && q / LOAD_EVERY < GROUP) {
        constexpr int n = q / LOAD_EVERY;
        if constexpr (n < LW) request_w(Int<n>{}, w_at, w_slot);
        else request_a(Int<(SET == 1 ? 0 : LA) + n - LW>{}, a_at, a_slot);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  int a_cur = 0, w_cur = 0;   // slots of the half at hand
  for (int s = 0; s < slabs; ++s) {
    const int w1 = w_cur + 1 == RW ? 0 : w_cur + 1, w2 = w1 + 1 == RW ? 0 : w1 + 1;
    const int a1 = a_cur + 1 == RA ? 0 : a_cur + 1, a_last = a_cur == 0 ? RA - 1 : a_cur - 1;
    half_step(Int<0>{}, a_cur, w1, w_half_at(2 * s + RW), w_cur, a_slab_at(s - 1 + RA), a_last);
    half_step(Int<1>{}, a1, w2, w_half_at(2 * s + 1 + RW), w1, a_slab_at(s + RA), a_cur);
    a_cur = a1, w_cur = w2;
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // the loads asked for beyond the last slab
  settle();

  const int row = lane % 16, quad = lane / 16;
  if constexpr (EPI == 3) {
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int m = m_base + (wm * WM + i) * 16 + row;
      if (m >= M) continue;
      float* p_row = partials + (static_cast<size_t>(blockIdx.z) * M + m) * N;
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const int n = (nt_base + tile_of(j)) * 16 + quad * 4;
        if (n < N) *reinterpret_cast<floatx4*>(p_row + n) = acc[i][j];
      }
    }
    return;
  }
  // The tile, rounded to bfloat16, through LDS: the stores are whole rows then, and the activation's code stands here once.
  constexpr int PITCH = NT * 16 + 8;   // elements
  static_assert(BM * PITCH <= RA * A_SLAB + RW * W_HALF, "the tile fits");
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0) & ~(15 << 8));
  bare_barrier();
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const uint2 packed{two_bf16(acc[i][j][0], acc[i][j][1]), two_bf16(acc[i][j][2], acc[i][j][3])};
      *reinterpret_cast<uint2*>(lds + ((wm * WM + i) * 16 + row) * PITCH + tile_of(j) * 16 + quad * 4) = packed;
    }
  __syncthreads();
  constexpr int PIECES = NT * 2 / (EPI == 1 ? 2 : 1);   // of eight outputs, in a row
  const int n_first = (EPI == 1 ? nt_base * 8 : nt_base * 16), rows_here = M - m_base < BM ? M - m_base : BM;
  auto store_rows = [&](auto&& value) __attribute__((always_inline)) {
#pragma unroll 2
    for (int p = threadIdx.x; p < rows_here * PIECES; p += 256) {
      const int r = p / PIECES, c = p % PIECES, n = n_first + c * 8;
      if (n >= (EPI == 1 ? N : NL)) continue;
      union Eight { uint4 q; uint32_t w[4]; } a, b, out;   // (pairs of bfloat16)
      const __bf16* from = lds + r * PITCH + (EPI == 1 ? (c / 2) * 32 + c % 2 * 8 : c * 8);
      a.q = *reinterpret_cast<const uint4*>(from);
      if (EPI == 1) b.q = *reinterpret_cast<const uint4*>(from + 16);
      else b = a;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        out.w[e] = two_bf16(value(__uint_as_float(a.w[e] << 16), __uint_as_float(b.w[e] << 16)),
                            value(__uint_as_float(a.w[e] & 0xffff0000u), __uint_as_float(b.w[e] & 0xffff0000u)));
      *reinterpret_cast<uint4*>(C + static_cast<size_t>(m_base + r) * ldc + n) = out.q;
    }
  };
  // (the rule's code once for each rule, not for each value)
  if constexpr (EPI == 1) {
    if (act == kActClampedGlu) store_rows([&](float g, float u) { return gated_product(kActClampedGlu, limit, g, u); });
    else if (act == kActSilu) store_rows([&](float g, float u) { return gated_product(kActSilu, limit, g, u); });
    else if (act == kActGeluTanh) store_rows([&](float g, float u) { return gated_product(kActGeluTanh, limit, g, u); });
    else store_rows([&](float g, float u) { return gated_product(act, limit, g, u); });
  } else {
    if (act == 0) store_rows([&](float x, float) { return x; });
    else if (act == 1 + kActSquaredRelu) store_rows([&](float x, float) { return gated_activation(kActSquaredRelu, x); });
    else store_rows([&](float x, float) { return gated_activation(act - 1, x); });
  }
}

template <int WM, int WN, int RA, int RW>
static void launch(const bf16* A, int64_t lda, const bf16* W, bf16* C, int64_t ldc, int M, int N, int K, int epi,
                   int act, float limit, int ks, float* partials, bool raw, Sections sec, hipStream_t stream) {
  constexpr int BM = 2 * WM * 16, BNW = 2 * WN * 16;
  const int NW = epi == 1 ? 2 * ((N + 15) / 16) * 16 : N;
  const int whole = sec.n_step > 0 ? (NW - 1) / sec.n_step : 0;   // sections before the last one
  const dim3 grid(whole * ((sec.n_step + BNW - 1) / BNW) + (NW - whole * sec.n_step + BNW - 1) / BNW, (M + BM - 1) / BM, ks);
  if (epi == 1)
    gemm_broad_kernel<WM, WN, RA, RW, 1><<<grid, 256, 0, stream>>>(A, lda, W, C, ldc, M, N, K, K / 32, act, limit, nullptr, sec);
  else if (raw)
    gemm_broad_kernel<WM, WN, RA, RW, 3><<<grid, 256, 0, stream>>>(A, lda, W, C, ldc, M, N, K, K / 32, act, limit, partials, sec);
  else
    gemm_broad_kernel<WM, WN, RA, RW, 0><<<grid, 256, 0, stream>>>(A, lda, W, C, ldc, M, N, K, K / 32, act, limit, nullptr, sec);
}

}  // namespace broad

// The tile (rows * 1000 + weight rows) and cut of K that this kernel is expected to be fastest with, and its microseconds: full
// rounds of 256 workgroups, and a last one whose slabs take the less time the fewer CUs have one (the clock rises), fitted to 27
// sizes of weights from 1,024 x 1,024 to 73,728 x 4,608 at 256 to 3,072 rows (3 to 6 % root mean square).  behind_us: what a cut costs the
// caller behind the product, beside the planes' bytes.
double gemm_broad_plan(int M, int N, int K, int epi, bool have_workspace, size_t workspace_bytes, int& tile, int& ks, double behind_us,
                       int n_step) {
  struct Tile { int rows, wrows; double alone, full, start; };   // us a slab alone and with every CU at work; us a round
  static const Tile tiles[4] = {{256, 288, 0.99, 1.45, 7.6}, {256, 256, 0.89, 1.35, 6.4}, {192, 288, 0.80, 1.19, 5.2}, {192, 256, 0.76, 1.05, 4.0}};
  const int NW = epi == 1 ? 2 * ((N + 15) / 16) * 16 : N, slabs = K / broad::BK;
  double best = -1.0;
  int cut_out = 1;
  for (const Tile& t : tiles) {
    const int columns = n_step > 0 ? NW / n_step * ((n_step + t.wrows - 1) / t.wrows) : (NW + t.wrows - 1) / t.wrows;   // (whole sections)
    const int64_t count = static_cast<int64_t>((M + t.rows - 1) / t.rows) * columns;
    const int cuts[3] = {ks > 1 ? ks : 1, static_cast<int>(broad::kCUs / count), static_cast<int>(2 * broad::kCUs / count)};
    for (int c = 0; c < 3; ++c) {
      const int cut = cuts[c];
      if (c > 0 && (ks > 1 || epi != 0 || cut < 2 || cut == cuts[c - 1] || cut > slabs / 4)) continue;
      const double partial_bytes = static_cast<double>(cut) * M * N * 4;
      if (cut > 1 && (!have_workspace || partial_bytes > static_cast<double>(workspace_bytes))) continue;
      const int64_t full = count * cut / broad::kCUs;
      const double rest = static_cast<double>(count * cut % broad::kCUs) / broad::kCUs;
      const int per = (slabs + cut - 1) / cut;
      double us = 3.0 + full * (per * t.full + t.start);
      if (rest > 0) us += per * (t.alone + (t.full - t.alone) * rest) + t.start;
      if (cut > 1) us += partial_bytes / 8e6 + partial_bytes / 5.5e6 + behind_us;   // written, and read again by whoever adds them up
      if (best < 0 || us < best) best = us, tile = t.rows * 1000 + t.wrows, cut_out = cut;
    }
  }
  ks = cut_out;
  return fmax(best, 5.0 + 2.0 * NW * K / 5.8e6);   // (the weights streamed once)
}

void gemm_broad(int tile, const void* A, int64_t lda, const void* W, void* C, int64_t ldc, int M, int N, int K, int epi,
                int act, float limit, int ks, float* partials, bool raw, Sections sec, hipStream_t stream) {
  const bf16* a = static_cast<const bf16*>(A);
  const bf16* w = static_cast<const bf16*>(W);
  bf16* c = static_cast<bf16*>(C);
  switch (tile) {
    case 256288: broad::launch<8, 9, 3, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, partials, raw, sec, stream); break;
    case 192288: broad::launch<6, 9, 3, 4>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, partials, raw, sec, stream); break;
    case 256256: broad::launch<8, 8, 3, 4>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, partials, raw, sec, stream); break;
    default: broad::launch<6, 8, 3, 4>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, partials, raw, sec, stream); break;
  }
}

}  // namespace sa
