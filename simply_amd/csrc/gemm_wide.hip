// C[M, N] = epilogue(A[M, K] . W[N, K]^T) in bfloat16 for very many rows (whole prompts), on tiles wide enough
// that the vector memory path is no longer the bound: the 128 x 128 tiles of the tiled kernel pull 96 KiB per
// slab of 64 columns through a CU's 64 bytes a clock, which caps it at about a third of the MFMA rate.
//
// A workgroup of eight waves (one per CU) owns 256 x 192, 256 x 128, 128 x 256 or 192 x 128 outputs (or one of four
// waves, two per CU, 128 x 192) and takes both operands through LDS, in slabs of 64 columns of K that go round two
// or three buffers, with loads that go from global memory straight into LDS (no registers in between).
//   * Layout in LDS: W as KiB blocks in MFMA operand order (16 rows x 32 columns, lane l holds row l % 16,
//     columns 8 (l / 16) ..), which is how it lies in global memory, so a block is a copy.  A as rows of 128 bytes
//     (eight lanes load a row: whole lines) whose eight 16-byte pieces are permuted by the row's number, so that
//     the 16 rows of a fragment read fall into different banks.  All fragment reads are ds_read_b128 without bank
//     conflicts (measured).
//   * Schedule of a wave: the fragments of the two halves of a slab have registers of their own; the products of
//     the second half are held back until after the next barrier, where they cover the fragment reads of the next
//     slab's first half, and the reads of the second half are covered by the products of the first: between two
//     barriers the MFMA unit always has products to do.  On the larger tiles the reads are issued one by one
//     between those products (a wave issues in order: many reads in a row keep its products back).  The loads of
//     the slab one or two ahead are spread over the products, one after every few: issued together after the
//     barrier, the waves queue up at the memory pipeline (16 cycles a load) while the MFMA unit idles; with two
//     buffers they all go out in the first half of a slab, so that the second half covers the last one's way.
//   * The products are taken transposed (W fragment as the first operand), so that a lane holds four neighbouring
//     columns of one row of C and stores them as one 8-byte piece.
//
// Epilogues: none; gated (C = act(A.Wg^T) * (A.Wu^T), both rounded to bfloat16 first, from one weight whose
// 16-row tiles alternate between Wg and Wu).  K must be a multiple of 64, N and ldc of 4.
//
// K may be cut over gridDim.z workgroups (a few hundred rows against a long K and few weight rows: too few tiles for
// 256 CUs otherwise): each writes its 32-bit partial tile to `partials` [z][M][N], and the tiled kernel's sum kernel
// adds them up.
#include "api.h"
#include "slabs.h"

namespace sa {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

namespace wide {

constexpr int BK = 64;
constexpr int kCUs = 256;  // compute units of an MI355X

using slabs::bare_barrier;
using slabs::waitcnt_vm;

// 16 bytes per lane from global memory (base + offset bytes, base the same for the whole wave) into LDS at byte
// address lds + 16 * lane (the same for the whole wave).  Written as an instruction: the compiler counts a load
// into LDS that it knows of as a pending LDS access for as long as the load is under way, and then makes every
// wait for a fragment read a wait for all of them.  It does not know of these loads: the kernel waits for them
// itself (vmcnt) before the barrier that precedes the first read of what they bring.
__device__ __forceinline__ void load_to_lds(const bf16* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(offset), "s"(base), "s"(lds)
               : "memory");
}

// Products of routed experts (ROUTED): row tile blockIdx.y is tile y of the sort kernel's plan (from plan[1 + 3 y] on: its
// expert, its first row in the sorted order, its rows), row m of it is row `sorted[first + m] / top` of A (by_token) or
// row first + m; W holds the experts' weights one behind the other, and w2, with the gated epilogue, the other factor's.
// EPI 0 and 1 write row first + m of C, EPI 4 the 32-bit product to row `sorted[first + m]` of `partials`.
struct Routed {
  const int* plan;
  const int* sorted;
  const bf16* w2;
  int by_token, top;
};
// EPI 4: row tiles from `tiles` on are those of a product beside the experts', rows of its own times one weight of as many outputs
// (the second product of a feed-forward that takes every token), bfloat16 results in the rows' order.
struct RoutedBeside : Routed {
  int tiles;
  const bf16* beside_a;
  const bf16* beside_w;
  bf16* beside_y;
  int64_t beside_lda, beside_ldc;
  int beside_k, beside_rows;
};

// (A launch's arguments hold what it reads and no more: 56 bytes of others in front of the grid's size cost 0.1 to 0.4 us a launch,
// 512 rows of 2,048 against 2,048 outputs 11.0 for 10.7.)
struct OneProduct {};
template <bool ROUTED, int EPI>
using Rows = std::conditional_t<!ROUTED, OneProduct, std::conditional_t<EPI == 4, RoutedBeside, Routed>>;
static_assert(std::is_empty_v<Rows<false, 0>> && sizeof(Rows<true, 1>) == 32, "what only some kernels read is an argument of those alone");

// WM x WN: 16 x 16 tiles of a wave (rows of A x rows of W); WAVES_M x (WAVES / WAVES_M) waves.
template <int WM, int WN, int WAVES_M, int EPI, int NSTAGE, int WAVES, bool ROUTED = false>
__global__ __launch_bounds__(WAVES * 64) void gemm_wide_kernel(const bf16* __restrict__ A, int64_t lda,
                                                        const bf16* __restrict__ W, bf16* __restrict__ C, int64_t ldc,
                                                        int M, int N, int K, int chunks, int act, float limit,
                                                        float* __restrict__ partials, Sections sec, Rows<ROUTED, EPI> rt) {
  constexpr int WAVES_N = WAVES / WAVES_M;
  constexpr int MT = WAVES_M * WM, NT = WAVES_N * WN;  // 16-row tiles of A and of W per workgroup
  constexpr int BM = MT * 16;
  constexpr int A_BLOCKS = MT * 2, W_BLOCKS = NT * 2;  // KiB blocks of a slab
  static_assert(A_BLOCKS % WAVES == 0 && W_BLOCKS % WAVES == 0, "every wave copies the same number of blocks");
  static_assert(EPI != 1 || WN % 2 == 0, "gate and factor tiles come in pairs");
  constexpr int APW = A_BLOCKS / WAVES, WPW = W_BLOCKS / WAVES;
  constexpr int STAGE = (A_BLOCKS + W_BLOCKS) * 512;  // elements
  __shared__ __attribute__((aligned(16))) __bf16 stages[NSTAGE * STAGE];
  const uint32_t lds_base = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) __bf16*)stages));

  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  // Which tile: workgroups go to the eight XCDs in turn, each with an L2 of its own; the numbering is turned round
  // so that an XCD gets a contiguous share of the tiles, and within it tiles go in columns eight wide, rows first.
  int bx = blockIdx.x, by = blockIdx.y;
  int row_first = 0, tile_rows = M;   // (ROUTED: the tile's rows)
  bool beside = false;
  if constexpr (ROUTED) {
    // (no turning round: how many tiles there are is known on the device only, and a tile's neighbours in x, which share
    // its rows, go to the XCDs in turn, so that an XCD meets the same weights again in the expert's next tile)
    if constexpr (EPI == 4) {
      beside = by >= rt.tiles;
      if (beside) {
        row_first = (by - rt.tiles) * BM, tile_rows = rt.beside_rows - row_first < BM ? rt.beside_rows - row_first : BM;
        A = rt.beside_a, lda = rt.beside_lda, W = rt.beside_w, K = rt.beside_k, chunks = K / 32;
        ldc = rt.beside_ldc;
      }
    }
    if (!beside) {
      if (by >= rt.plan[0]) return;
      row_first = rt.plan[2 + 3 * by], tile_rows = rt.plan[3 + 3 * by];
      const size_t expert = static_cast<size_t>(rt.plan[1 + 3 * by]) * ((N + 15) / 16) * chunks * 512;
      W += expert;
      if (EPI == 1) rt.w2 += expert;
    }
  } else {
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
  // this workgroup's share of K: slabs slab0 .. slab0 + slabs
  const int slabs_all = K / BK;
  const int slab0 = static_cast<int>(static_cast<int64_t>(blockIdx.z) * slabs_all / gridDim.z);
  const int slabs = static_cast<int>(static_cast<int64_t>(blockIdx.z + 1) * slabs_all / gridDim.z) - slab0;
  A += static_cast<size_t>(slab0) * BK;
  const int m_base = ROUTED ? 0 : by * BM;
  const int NW = EPI == 1 ? 2 * ((N + 15) / 16) * 16 : N;
  // several products at once: which section this workgroup is in, its columns of A, its rows of W
  int first_tile = 0, NL = NW;   // the section's first 16-row tile of W and the end of its rows
  if (sec.n_step > 0) {
    constexpr int BNW = NT * 16;
    const int per = (sec.n_step + BNW - 1) / BNW, s = bx / per;
    bx -= s * per;
    first_tile = s * (sec.n_step / 16);
    A += static_cast<size_t>(s) * sec.a_step;
    NL = (s + 1) * sec.n_step < NW ? (s + 1) * sec.n_step : NW;
  }
  const int ntiles = (NL + 15) / 16;
  const int nt_base = first_tile + bx * NT;

  // ---- what this wave copies of every slab: KiB blocks wave + WAVES i of A and of W.
  // A block b is rows 8 (b % 2) .. + 8 of tile b / 2, all 64 columns of the slab: eight lanes per row read its 128
  // bytes, so a load is eight whole lines.  In LDS a row's eight 16-byte pieces are permuted (piece p of row r of
  // the tile lies at p ^ (r / 2)), which makes the fragment reads below (16 rows, one piece each) hit all banks.
  // W block b is tile b / 2, columns 32 (b % 2) .. of the slab: a KiB as it lies in global memory.
  // Rows beyond M read row M - 1, tiles beyond the last the last one (their products are never stored).
  const int half_mine = wave % 2, tile_mine = wave / 2;
  uint32_t a_off[APW];  // bytes; the host checks that M * lda fits
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    const int r = half_mine * 8 + lane / 8;  // row of the tile
    const int m = m_base + (tile_mine + (WAVES / 2) * i) * 16 + r;
    int from = m < tile_rows ? m : tile_rows - 1;
    if constexpr (ROUTED) from = rt.by_token ? rt.sorted[row_first + from] / rt.top : row_first + from;
    a_off[i] = (static_cast<uint32_t>(from) * static_cast<uint32_t>(lda) + ((lane % 8) ^ (r / 2)) * 8) * 2;
  }
  const bf16* w_from[WPW];  // the same for the whole wave
#pragma unroll
  for (int i = 0; i < WPW; ++i) {
    const int nt = nt_base + tile_mine + (WAVES / 2) * i;
    const int clamped = __builtin_amdgcn_readfirstlane(nt < ntiles ? nt : ntiles - 1);
    // (routed gated products: the two factors' tiles alternate here, but lie in weights of their own)
    const bf16* from = W;
    if constexpr (ROUTED && EPI == 1) from = clamped % 2 ? rt.w2 : W;
    const int at = ROUTED && EPI == 1 ? clamped / 2 : clamped;
    w_from[i] = from + (static_cast<size_t>(at) * chunks + half_mine) * 512 + static_cast<size_t>(slab0) * 1024;
  }
  // load n (of LOADS) of slab `slab` into buffer `buf`
  constexpr int LOADS = APW + WPW;
  auto request_one = [&](int n, int slab, int buf) __attribute__((always_inline)) {
    const uint32_t to = lds_base + static_cast<uint32_t>(buf) * (STAGE * 2);
    if (n < APW)
      load_to_lds(A + static_cast<size_t>(slab) * BK, a_off[n], to + ((tile_mine + (WAVES / 2) * n) * 2 + half_mine) * 1024);
    else
      load_to_lds(w_from[n - APW] + static_cast<size_t>(slab) * 1024, lane * 16,
                  to + (A_BLOCKS + (tile_mine + (WAVES / 2) * (n - APW)) * 2 + half_mine) * 1024);
  };

  floatx4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // this lane's piece of an A fragment (row lane % 16, columns 32 kc + 8 (lane / 16) ..) within its tile, elements
  int a_frag[2];
#pragma unroll
  for (int kc = 0; kc < 2; ++kc) {
    const int r = lane % 16;
    a_frag[kc] = r * 64 + ((kc * 4 + lane / 16) ^ (r / 2)) * 8;
  }
  // Fragments of the two halves of a slab (columns 0 .. 31 and 32 .. 63) in registers of their own.  The products
  // of the second half are held back until after the next barrier, where they cover the time that the fragment
  // reads of the next slab's first half take; the reads of the second half are covered by the products of the
  // first.  So the MFMA unit always has products to do while LDS reads are under way.
  bf16x8 fa[2][WM], fw[2][WN];
  auto read = [&](const __bf16* stage, int kc) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
      fa[kc][i] = *reinterpret_cast<const bf16x8*>(stage + (wm * WM + i) * 1024 + a_frag[kc]);
#pragma unroll
    for (int j = 0; j < WN; ++j)
      fw[kc][j] = *reinterpret_cast<const bf16x8*>(stage + ((A_BLOCKS + (wn * WN + j) * 2 + kc) * 64 + lane) * 8);
  };
  // fragment n of half kc alone: W's first (the first row of products needs them all), then A's
  auto read_one = [&](const __bf16* stage, int kc, int n) __attribute__((always_inline)) {
    if (n < WN)
      fw[kc][n] = *reinterpret_cast<const bf16x8*>(stage + ((A_BLOCKS + (wn * WN + n) * 2 + kc) * 64 + lane) * 8);
    else
      fa[kc][n - WN] = *reinterpret_cast<const bf16x8*>(stage + (wm * WM + n - WN) * 1024 + a_frag[kc]);
  };
  // Tiles with enough products read the fragments of the other half one by one, each after one of the first
  // products of this half, instead of all of them before: a wave issues in order, and sixteen reads in a row keep
  // its products from the MFMA unit for a few hundred cycles.
  constexpr bool INTERLEAVED = WM * WN >= 2 * (WM + WN);
  // The products of half kc (`first`: 0 for the held-back half, which comes first after the barrier; 1 for the
  // other; -1: no loads).  After every EVERY products, counted through the slab, one load of slab `slab` is asked
  // for: spread out, so that the waves do not queue up at the memory pipeline (which takes 16 cycles for each) while
  // the MFMA unit idles, and early: with two buffers all of them among the first half's products, so that the
  // second half's cover the time that the last one takes.
  constexpr int SPAN = NSTAGE == 2 ? WM * WN : 2 * WM * WN;
  constexpr int EVERY = SPAN / LOADS > 0 ? SPAN / LOADS : 1;
  constexpr int PER = SPAN / LOADS > 0 ? 1 : (LOADS + SPAN - 1) / SPAN;  // (small tiles: several loads after each product)
  auto multiply = [&](int kc, int first, int slab, int buf, const __bf16* rstage = nullptr, int rkc = -1)
                      __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WM; ++i) {
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[kc][j], fa[kc][i], acc[i][j], 0, 0, 0);
        if (INTERLEAVED && rkc >= 0 && i * WN + j < WM + WN) {
          __builtin_amdgcn_sched_barrier(0);
          read_one(rstage, rkc, i * WN + j);
          __builtin_amdgcn_sched_barrier(0);
        }
        const int q = (first > 0 ? WM * WN : 0) + i * WN + j + 1;  // products of this slab so far
#pragma unroll
        for (int e = 0; e < PER; ++e) {
          const int n = (q / EVERY - 1) * PER + e;
          if (first >= 0 && q % EVERY == 0 && n < LOADS) {
            __builtin_amdgcn_sched_barrier(0);
            request_one(n, slab, buf);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
  };
  // The slabs go round NSTAGE buffers.  Before the barrier of slab s this wave's loads of slab s have arrived (those
  // of the NSTAGE - 2 slabs after it may be under way) and its fragment reads of slab s - 1 are done; after it
  // everyone's, so that the loads of slab s + NSTAGE - 1 may go into the buffer of slab s - 1.  Past the last slab
  // the last one is loaded again (no branch).
#pragma unroll
  for (int p = 0; p < NSTAGE; ++p)
#pragma unroll
    for (int n = 0; n < LOADS; ++n) request_one(n, p < slabs ? p : slabs - 1, p);
  // (routed) A wave none of whose rows exist copies its share of every slab and leaves the matrix units to the others.
  if (ROUTED && wm * WM * 16 >= tile_rows) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm((NSTAGE - 1) * LOADS));
    bare_barrier();
    int into = 0;
    for (int s = 1; s < slabs; ++s) {
      __builtin_amdgcn_s_waitcnt(waitcnt_vm((NSTAGE - 2) * LOADS));
      bare_barrier();
      const int ahead = s + NSTAGE - 1 < slabs ? s + NSTAGE - 1 : slabs - 1;
#pragma unroll
      for (int n = 0; n < LOADS; ++n) request_one(n, ahead, into);
      into = into + 1 == NSTAGE ? 0 : into + 1;
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    return;
  }
  // slab 0: nothing held back yet, and its loads for later are already asked for
  __builtin_amdgcn_s_waitcnt(waitcnt_vm((NSTAGE - 1) * LOADS));
  bare_barrier();
  read(stages, 0);
  read(stages, 1);
  __builtin_amdgcn_sched_barrier(0);
  multiply(0, -1, 0, 0);
  int cur = 1, target = 0;
  for (int s = 1; s < slabs; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm((NSTAGE - 2) * LOADS) & ~(15 << 8));
    bare_barrier();
    const int ahead = s + NSTAGE - 1 < slabs ? s + NSTAGE - 1 : slabs - 1;
    const __bf16* stage = stages + cur * STAGE;
    if (INTERLEAVED) {
      multiply(1, 0, ahead, target, stage, 0);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, 1, ahead, target, stage, 1);
    } else {
      read(stage, 0);
      __builtin_amdgcn_sched_barrier(0);
      multiply(1, 0, ahead, target);
      __builtin_amdgcn_sched_barrier(0);  // (reads moved up among these products would need registers of their own)
      read(stage, 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, 1, ahead, target);
    }
    target = cur;
    cur = cur + 1 == NSTAGE ? 0 : cur + 1;
  }
  multiply(1, -1, 0, 0);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // the loads asked for beyond the last slab

  // ---- epilogue.  acc[i][j][v] is the product at row (tile i, lane % 16) of A and row (tile j, 4 (lane / 16) + v)
  // of W.
  const int row = lane % 16, quad = lane / 16;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int m = m_base + (wm * WM + i) * 16 + row;
    if (m >= tile_rows) continue;
    if constexpr (EPI == 4) {
      if (beside) {   // (rounded, in the rows' order)
        bf16* c_row = rt.beside_y + static_cast<size_t>(row_first + m) * ldc;
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          const int n = (nt_base + wn * WN + j) * 16 + quad * 4;
          uint2 packed;
          packed.x = static_cast<uint32_t>(float_to_bf16(acc[i][j][0]).bits) | (static_cast<uint32_t>(float_to_bf16(acc[i][j][1]).bits) << 16);
          packed.y = static_cast<uint32_t>(float_to_bf16(acc[i][j][2]).bits) | (static_cast<uint32_t>(float_to_bf16(acc[i][j][3]).bits) << 16);
          if (n < NL) *reinterpret_cast<uint2*>(c_row + n) = packed;
        }
        continue;
      }
      float* y_row = partials + static_cast<size_t>(rt.sorted[row_first + m]) * ldc;
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const int n = (nt_base + wn * WN + j) * 16 + quad * 4;
        if (n < NL) *reinterpret_cast<floatx4*>(y_row + n) = acc[i][j];
      }
      continue;
    }
    if (EPI == 3) {  // this workgroup's share of the sum, as it is
      float* p_row = partials + (static_cast<size_t>(blockIdx.z) * M + m) * N;
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const int n = (nt_base + wn * WN + j) * 16 + quad * 4;
        if (n < NL) *reinterpret_cast<floatx4*>(p_row + n) = acc[i][j];
      }
      continue;
    }
    bf16* c_row = C + static_cast<size_t>(row_first + m) * ldc;
    constexpr int OUT = EPI == 1 ? WN / 2 : WN;
#pragma unroll
    for (int j = 0; j < OUT; ++j) {
      const int tile = EPI == 1 ? (nt_base + wn * WN) / 2 + j : nt_base + wn * WN + j;
      const int n = tile * 16 + quad * 4;
      if (n >= (EPI == 1 ? N : NL)) continue;
      float x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (EPI == 1)
          x[v] = gated_product(act, limit, to_float(float_to_bf16(acc[i][2 * j][v])),
                               to_float(float_to_bf16(acc[i][2 * j + 1][v])));
        else
          x[v] = acc[i][j][v];
        // (without another epilogue, act > 0 asks for the activation act - 1 of the product rounded to bfloat16)
        if (EPI == 0 && act > 0) x[v] = gated_activation(act - 1, to_float(float_to_bf16(x[v])));
      }
      uint2 packed;
      packed.x = static_cast<uint32_t>(float_to_bf16(x[0]).bits) | (static_cast<uint32_t>(float_to_bf16(x[1]).bits) << 16);
      packed.y = static_cast<uint32_t>(float_to_bf16(x[2]).bits) | (static_cast<uint32_t>(float_to_bf16(x[3]).bits) << 16);
      *reinterpret_cast<uint2*>(c_row + n) = packed;
    }
  }
}

template <int WM, int WN, int WAVES_M, int NSTAGE, int WAVES = 8>
static void launch(const bf16* A, int64_t lda, const bf16* W, bf16* C, int64_t ldc, int M, int N, int K, int epi,
                   int act, float limit, int ks, float* partials, bool raw, Sections sec, hipStream_t stream) {
  constexpr int BM = WAVES_M * WM * 16, BNW = (WAVES / WAVES_M) * WN * 16;
  const int NW = epi == 1 ? 2 * ((N + 15) / 16) * 16 : N;
  const int whole = sec.n_step > 0 ? (NW - 1) / sec.n_step : 0;   // sections before the last one
  const dim3 grid(whole * ((sec.n_step + BNW - 1) / BNW) + (NW - whole * sec.n_step + BNW - 1) / BNW, (M + BM - 1) / BM, ks);
  if (epi == 1)
    gemm_wide_kernel<WM, WN, WAVES_M, 1, NSTAGE, WAVES><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, C, ldc, M, N, K, K / 32,
                                                                                         act, limit, nullptr, sec, {});
  else if (raw)
    gemm_wide_kernel<WM, WN, WAVES_M, 3, NSTAGE, WAVES><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, C, ldc, M, N, K, K / 32,
                                                                                         act, limit, partials, sec, {});
  else
    gemm_wide_kernel<WM, WN, WAVES_M, 0, NSTAGE, WAVES><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, C, ldc, M, N, K, K / 32,
                                                                                         act, limit, nullptr, sec, {});
}

template <int WM, int WN, int WAVES_M, int NSTAGE, int WAVES>
static void launch_routed(const bf16* A, int64_t lda, const bf16* W, const RoutedBeside& rt, bf16* C, float* y, int64_t ldc, int tiles,
                          int rows, int N, int K, int act, float limit, hipStream_t stream) {
  constexpr int BNW = (WAVES / WAVES_M) * WN * 16;
  const int NW = rt.w2 != nullptr ? 2 * ((N + 15) / 16) * 16 : N;
  constexpr int BM = WAVES_M * WM * 16;
  const dim3 grid((NW + BNW - 1) / BNW, tiles + (rt.beside_rows + BM - 1) / BM);
  if (rt.w2 != nullptr)
    gemm_wide_kernel<WM, WN, WAVES_M, 1, NSTAGE, WAVES, true><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, C, ldc, rows, N, K, K / 32,
                                                                                               act, limit, nullptr, Sections{}, rt);
  else if (y != nullptr)
    gemm_wide_kernel<WM, WN, WAVES_M, 4, NSTAGE, WAVES, true><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, C, ldc, rows, N, K, K / 32,
                                                                                               0, 0.f, y, Sections{}, rt);
  else
    gemm_wide_kernel<WM, WN, WAVES_M, 0, NSTAGE, WAVES, true><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, C, ldc, rows, N, K, K / 32,
                                                                                               act, limit, nullptr, Sections{}, rt);
}

}  // namespace wide

// Products of routed experts on this kernel's tiles: 64 rows of an expert x 128 weight rows with three buffers, two workgroups of four
// waves a CU, or (tile_rows) 128 x 256 with three, one of eight waves, 64 x 64 outputs each: a tile's upper 64 rows, which an expert's
// last tile often lacks, are the business of four waves of their own, that then leave the matrix units to the others.  Gate and up
// together with down of 16 experts, in microseconds:
//   2,048 x 2,048, rows an expert   37: 89 / 100   64: 105 / 95    96: 106 / 99    128: 127 / 120   256: 186 / 173   400: 254 / 206 (64 / 128)
//   4,096 x 3,584                   64: 304 / 275  96: 339 / 283   136: 431 / 437  256: 600 / 534   400: 907 / 711
//   3,072 x 2,048                   68: 149 / 130  96: 157 / 137   136: 199 / 207  256: 275 / 248   512: 492 / 388
//   2,048 x 3,072                   68: 143 / 147  96: 151 / 154   136: 192 / 185  256: 274 / 243   512: 477 / 392
//   2,560 x 2,560                   68: 168 / 159  96: 187 / 168   136: 223 / 243  256: 298 / 287   512: 508 / 436
//   3,072 x 1,536                   68: 110 / 101  136: 157 / 187  272: 226 / 251  336: 263 / 253   512: 362 / 317
//   1,024 x 4,096                   60: 94 / 116   96: 110 / 128   136: 145 / 149  208: 172 / 167   336: 239 / 214
//   4,096 x 1,024                   60: 111 / 106  96: 109 / 115   136: 138 / 146  240: 188 / 195   336: 237 / 199
//   1,024 x 8,192                   60: 180 / 235  128: 265 / 271  192: 318 / 298  256: 413 / 354
//   2,048 x 1,536                   60: 79 / 79    128: 99 / 106   256: 146 / 152  400: 200 / 170
//   1,792 x 1,792                   60: 73 / 78    128: 129 / 115  256: 178 / 178  400: 232 / 242
//   1,536 x 1,536                   60: 59 / 63    128: 83 / 88    256: 122 / 115  400: 159 / 162
//   1,024 x 1,024                   60: 37 / 43    128: 48 / 48    256: 67 / 68    400: 88 / 73
// (128 x 192 of four waves, two a CU, which the 128 rows were before: 209 at 256 rows of 2,048 x 2,048, 626 of 4,096 x 3,584.)  Also
// tried for 64 rows: eight waves with six buffers, 64 x 256, four waves across; for 128: 128 x 128 (191 and 546), waves of 128 x 64 and
// 64 x 128 (237 and 233).
bool gemm_wide_routed_takes(int N, int K, int64_t lda, int64_t a_rows, int64_t ldc, const void* A, const void* W, const void* W2,
                            const void* C, int tile_rows) {
  auto aligned = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
  return (tile_rows == 64 || tile_rows == 128) && K % wide::BK == 0 && N % 4 == 0 && lda % 8 == 0 && ldc % 4 == 0 && aligned(A, 16) &&
         aligned(W, 16) && aligned(W2, 16) && aligned(C, 16) && a_rows * lda < (int64_t{1} << 31);
}

// act: the gated rule, or with one weight and a bfloat16 result 1 + the activation.  y (and no C): the 32-bit product, a row
// per pair.
int gemm_wide_routed(const void* A, int64_t lda, const void* W, const void* W2, void* C, float* y, int64_t ldc, int tiles, int N,
                     int K, int tile_rows, const int* plan, const int* sorted, int by_token, int top, int act, float limit,
                     hipStream_t stream, const void* beside_a, int64_t beside_lda, const void* beside_w, void* beside_y,
                     int64_t beside_ldc, int beside_k, int beside_rows) {
  wide::RoutedBeside rt;
  rt.plan = plan, rt.sorted = sorted, rt.w2 = static_cast<const bf16*>(W2), rt.by_token = by_token, rt.top = top;
  rt.tiles = tiles, rt.beside_a = static_cast<const bf16*>(beside_a), rt.beside_w = static_cast<const bf16*>(beside_w);
  rt.beside_y = static_cast<bf16*>(beside_y), rt.beside_lda = beside_lda, rt.beside_ldc = beside_ldc, rt.beside_k = beside_k, rt.beside_rows = beside_rows;
  const bf16* a = static_cast<const bf16*>(A);
  const bf16* w = static_cast<const bf16*>(W);
  bf16* c = static_cast<bf16*>(C);
  if (tile_rows == 128) wide::launch_routed<4, 4, 2, 3, 8>(a, lda, w, rt, c, y, ldc, tiles, tile_rows, N, K, act, limit, stream);
  else wide::launch_routed<2, 4, 2, 3, 4>(a, lda, w, rt, c, y, ldc, tiles, tile_rows, N, K, act, limit, stream);
  return check_launch("gemm_wide_routed");
}

bool gemm_wide_takes(int M, int N, int K, int64_t lda, int64_t ldc, const void* A, const void* W, const void* W2,
                     const void* C, int c_dtype, int epi, int packed) {
  auto aligned = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
  return packed && W2 == nullptr && (epi == 0 || epi == 1) && M >= 1 &&
         (c_dtype == kBF16 || (c_dtype == kF32 && epi == 0 && ldc == N && M > 64 && N >= 512 && aligned(C, 16))) && K % wide::BK == 0 &&
         N % 4 == 0 && lda % 8 == 0 && ldc % 4 == 0 && aligned(A, 16) && aligned(W, 16) && aligned(C, 8) &&
         static_cast<int64_t>(M) * lda < (int64_t{1} << 31);  // byte offsets of rows are kept in 32 bits
}

// Of a tile of 32,768 outputs with every CU at work.
double gemm_wide_tile_us(int K) { return 0.78 * K / wide::BK + 2.8; }

// The time of an uncut product on tiles of `shape`, `columns` of them side by side: their rounds of slabs at what 128 outputs of 256 rows (or
// as many of another tile) take, fitted like the broad kernel's.  (128 x 128, which take longer for their size, are taken for few tiles, at
// which the clock is higher: 0.69 to 0.98 us there.)
static double rounds_us(int shape, int M, int64_t columns, int NW, int K, int epi) {
  const int rows = shape / 1000 % 1000, wrows = shape % 1000;
  const int64_t rounds = ((M + rows - 1) / rows * columns + wide::kCUs - 1) / wide::kCUs;
  return fmax(5.0 + 2.0 * NW * K / 5.8e6, 3.0 + rounds * ((epi == 1 ? 0.88 : 0.78) * (K / wide::BK) * rows * wrows / 32768.0 + 2.8));
}

// The tile and the cut of K for a product whose caller fixes neither, and the time that this kernel is expected to
// take with them in microseconds (the figure by which the library chooses between its product kernels).
static double plan_shape(int M, int N, int K, int epi, bool have_workspace, size_t workspace_bytes, int& shape, int& ks, bool planes, bool broad = true) {
  const int NW_all = epi == 1 ? 2 * ((N + 15) / 16) * 16 : N;
  const int asked = ks;   // the caller's cut of K, 1: none
  // without a fitted model below: the weights streamed once at the rate this kernel reaches for few rows, or the
  // products at its rate for many, whichever takes longer, after its start
  double us = 5.0 + 0.02 * (M < 64 ? M : 64) +
              fmax(2.0 * NW_all * K / 5.8e6, static_cast<double>(M) * NW_all * K / (1.05e9 / 2));
  // The cost of a shape: the workgroups that the busiest CU gets times the size of the tile; of equals the first.
  // Workgroups of four waves run two to a CU, where one's epilogue and first loads overlap the other's
  // products (measured: 7-9 % faster than one workgroup of twice the tile once every CU has two of them;
  // slower when it has one; from one and a half per CU on it is also the best for few rows of very many weight
  // rows, which are bound by streaming them).  A tile of 128 x 128, whose waves read more of LDS for a product, takes
  // 1.38 times as long for its size, so it is taken in two cases alone.  One round of it is cheaper than one of 192 x 128, however few
  // tiles that is; measured, us, at 16 to 256 tiles of gated products of 129 to 4,096 rows and 104 to 256 of plain ones of 1,537 to
  // 4,096: ahead in all 96, by 3 to 38 % (2,048 rows against 2,048 outputs of K = 2,048 20.8 for 23.7, of 8,192 75.5 for 78.5; 1,024 of
  // 4,096 28.3 for 35.0; gated, 129 rows against 512 of 1,024 11.8 for 14.5, 256 against 1,024 of 4,096 37.5 for 38.9, 256
  // against 8,192 of 2,048 27.2 for 30.1).  And two rounds of it than one of 256 x 192 (1,664 rows against 4,992 outputs 44.5 for
  // 46.4); a second round costs more than one of 192 x 128 (2,048 rows against 2,304 outputs: 35 for 25).
  const int NW = epi == 1 ? 2 * ((N + 15) / 16) * 16 : N;
  const int shapes[6][4] = {{2128192, 128, 192, 93}, {2256192, 256, 192, 100}, {3256128, 256, 128, 100},
                            {3128256, 128, 256, 100}, {3192128, 192, 128, 100}, {4128128, 128, 128, 138}};
  int64_t best = -1;
  for (const auto& sh : shapes) {
    const int64_t tiles = static_cast<int64_t>((M + sh[1] - 1) / sh[1]) * ((NW + sh[2] - 1) / sh[2]);
    if (sh[3] < 100 && tiles < wide::kCUs * 3 / 2) continue;
    const int64_t cost = ((tiles + wide::kCUs - 1) / wide::kCUs) * sh[1] * sh[2] * sh[3];
    if (best < 0 || cost < best) {
      best = cost;
      shape = sh[0];
    }
  }
  // A gated product of few rows whose tiles of 128 weight rows make one round at most (the 2B and 9B feed-forward
  // for up to 128 decoding requests) streams its weights: rows of 64 (or 128) with the deepest pipeline that fits
  // are 5 to 25 % faster there than the large tiles (2B at 64 rows: 23 against 28 us; 9B: 39 against 48).
  if (epi == 1 && M <= 128) {
    const int rows = M <= 64 ? 64 : 128;
    if (static_cast<int64_t>((M + rows - 1) / rows) * ((NW + 127) / 128) <= wide::kCUs) shape = M <= 64 ? 6064128 : 3128128;
  }
  // 17 to 1,536 rows without an epilogue (portions of prompts, many decoding requests): the tiles above are too few
  // for 256 CUs, and every workgroup walks all of K at the pace of its own slabs.  Smaller tiles with deeper
  // pipelines, and K cut over workgroups so that about one round of them covers the GPU, chosen by a model of the
  // time fitted to measurements at the 2B, 9B and 27B sizes (64 to 2,048 rows, seven tiles, one to fourteen cuts;
  // it is within 6 % of the best measured choice nearly everywhere, and a fifth faster in sum than either the
  // uncut tiles above or the tiled kernel with its cut: the 2B down projection at 512 rows takes 36 us against 55).
  // More rows against few outputs (64 tiles of 128 x 128 at most) too: 2,048 rows of K = 4,096 against 512 outputs 27.6 / 15.2 us, of K =
  // 2,048 against 256 16.5 / 10.9 and against 64 15.5 / 13.4, 3,000 of 2,304 against 160 17.2 / 11.1 (uncut / with the cut).
  const bool few_tiles = static_cast<int64_t>((M + 127) / 128) * ((N + 127) / 128) <= 64;
  if (epi == 0 && (M <= 1536 || few_tiles)) {  // (fewer than 17 rows come here only against a very long K)
    struct Tile { int code, rows, wrows; double eff, start; };  // share of the MFMA rate in the loop; us to start
    static const Tile tiles[7] = {{3128128, 128, 128, 0.425, 1.44}, {3128256, 128, 256, 0.535, 2.03},
                                  {3192128, 192, 128, 0.535, 1.25}, {3256128, 256, 128, 0.615, 1.58},
                                  {5128064, 128, 64, 0.326, 0.85},  {6064064, 64, 64, 0.234, 0.80},
                                  {6064128, 64, 128, 0.277, 1.08}};
    const int slabs = K / wide::BK;
    double best_us = -1.0;
    int best_ks = 1;
    for (const Tile& t : tiles) {
      const int64_t count = static_cast<int64_t>((M + t.rows - 1) / t.rows) * ((N + t.wrows - 1) / t.wrows);
      const int cuts[3] = {1, static_cast<int>(wide::kCUs / count), static_cast<int>(2 * wide::kCUs / count)};
      for (int c = 0; c < 3; ++c) {
        const int cut = cuts[c];
        if (cut < 1 || (c > 0 && (cut < 2 || cut == cuts[c - 1])) || cut > slabs / 4) continue;
        const double partial_bytes = static_cast<double>(cut) * M * N * 4;
        if (cut > 1 && (!have_workspace || partial_bytes > static_cast<double>(workspace_bytes))) continue;
        const int64_t rounds = (count * cut + wide::kCUs - 1) / wide::kCUs;
        const int per = (slabs + cut - 1) / cut;
        // a CU's MFMA rate: 4.9 M multiply-adds of bfloat16 a microsecond
        double us = rounds * (static_cast<double>(per) * t.rows * t.wrows * wide::BK / (4.9e6 * t.eff) + t.start) + 3.2;
        if (cut > 1) us += partial_bytes / 5.5e6 + partial_bytes / 4.9e6 + 3.7;  // written, read again, the sum kernel
        if (best_us < 0 || us < best_us) {
          best_us = us;
          shape = t.code;
          best_ks = cut;
        }
      }
    }
    if (ks == 1) ks = best_ks;
    // (the model of the tiles knows nothing of memory: the weights streamed once from HBM are a floor under it)
    if (best_us >= 0) us = fmax(best_us, 5.0 + 0.02 * (M < 64 ? M : 64) + 2.0 * NW_all * K / 5.8e6);
  }
  // The tiles of the broad kernel against all of these.  What the others take beyond 1,536 rows or gated, where no model above
  // says it: rounds_us.
  // (Behind other kernels, weights in HBM, the broad tiles keep their time better than in a loop of the one product, by which both are
  // fitted: 2,048 rows against 6,144 outputs of K = 2,048 49 and 49 us there, 60 and 49 in a prompt.  Hence the line at 1.03; at 1.12
  // prompts are 0.3 to 1 % slower again.)
  if (broad && M >= 96) {
    const bool fitted = epi == 0 && (M <= 1536 || few_tiles);
    double best_us = fitted ? us : rounds_us(shape, M, (NW + shape % 1000 - 1) / (shape % 1000), NW_all, K, epi);
    // With the cut that the tiles above take, or where they take none any.  (More than three cuts of few rows cost more than the broad
    // kernel's model says: 160 rows of 9,216 against 2,304 outputs with 14 cuts 23 and 28 us, 896 with four 49 and 56, 129 of 8,192
    // against 2,048 with 16 20 and 24, all expected at about the same.)
    // Beyond 1,536 rows the tiles above are not cut: where the sum is a kernel of its own, it counts, and cuts are taken only ahead (3,072 rows
    // of 9,216 against 2,304 outputs in two cuts 112 / 115 us with the sum, 132 / 127 with a norm that adds them up, 4,096 of 16,384 against
    // 2,048 207 / 219 and 230 / 229); five and more only well ahead and of 13 slabs or more each, either way (1,600 of 4,096 against 1,024 in
    // seven 28 / 32, of 4,608 against 640 in nine 31 / 33, 1,800 of 6,144 against 1,280 in five 42 / 53 and 52 / 59; of 8,192 against 1,024 in
    // six 52 / 46, 2,500 against 512 in nine 50 / 38, 2,047 of 36,864 against 640 in ten 282 / 103).  The
    // pass for an activation behind a cut does not count: it takes what the code in an uncut product's epilogue takes (2,304 outputs of
    // 9,216, erf GELU, 4,096 rows: 18 us and 19).
    const double behind_us = fitted || planes ? 0.0 : 3.7;
    const int others = ks;
    int tile = 0, cut = others;
    const double broad_us = gemm_broad_plan(M, N, K, epi, have_workspace, workspace_bytes, tile, cut, behind_us);
    const double line = cut == 1 ? 1.03 : fitted ? (cut > 3 ? 0.94 : 1.03) : cut > 4 ? (K / wide::BK / cut >= 13 ? 0.93 : 0.0) : planes ? 1.03 : 0.96;
    if (broad_us < line * best_us) {
      shape = 1000000 + tile;
      ks = cut;
      best_us = broad_us;
      // (the figure that the other kernels' are compared with, crude as theirs, never grows by a better tile: 4,096 rows of K = 64 against
      // 14,336 gated outputs would go to the tiled kernel, 125 us for 72)
      us = fmin(us, broad_us);
    }
    // With a cut of their own beside tiles that are cut too, which was found for tiles of another size, only well ahead: 544 rows of 36,864
    // against 4,608 outputs 216 / 178 us, 640 261 / 217, of 14,336 against 6,144 320 rows 87 / 76, against 4,096 544 rows 85 / 76.  Of 80
    // sizes that the model has up to 8 % ahead or behind 61 were slower (129 rows of 4,096 against 12,288, by the model 7 % ahead, by 14 %).
    if (asked == 1 && others > 1) {
      int own_tile = 0, own_cut = 1;
      const double own_us = gemm_broad_plan(M, N, K, epi, have_workspace, workspace_bytes, own_tile, own_cut, behind_us);
      if (own_cut > 1 && own_us < 0.92 * best_us) {
        shape = 1000000 + own_tile;
        ks = own_cut;
        us = fmin(us, own_us);
      }
    }
  }
  return us;
}

// Several products at once (sections of n_step outputs, 0: one product): the broad kernel's tile for the whole sections where they on it and
// a shorter last one by itself (at 2,047 rows of four sections of 2,048 outputs it would be eight more tiles behind a full round) are
// ahead of the wide kernel's `shape` and cut of K, whose time is planned_us; else 0, as where no section is whole.  Measured, us, wide / broad
// and the rest: 2,047 rows of four sections of 2,048 and 64 outputs 78 / 63, of three and 16 55 / 56, 1,031 rows of four 49 / 46, 4,096
// 140 / 120; sections of 4,096, 700 rows 108 / 89, 1,024 without a rest 125 / 112, 2,500 334 / 284; of 1,024, 3,000 rows 45 / 31, 4,096
// without a rest 42 / 34.
static int sections_broad_tile(int M, int N, int K, int n_step, bool have_workspace, size_t workspace_bytes, int shape, int ks, double planned_us) {
  if (n_step <= 0 || N < n_step || M < 96) return 0;
  const int whole = N / n_step, rest = N % n_step;
  int tile = 0, one = 1;
  double us = gemm_broad_plan(M, whole * n_step, K, 0, false, 0, tile, one, 0.0, n_step);
  if (rest > 0) us += fmin(gemm_tiled_predict_us(M, rest, K, 0), gemm_wide_predict_us(M, rest, K, 0, have_workspace, workspace_bytes, false));
  const int wrows = shape % 1000;
  const int64_t columns = static_cast<int64_t>(whole) * ((n_step + wrows - 1) / wrows) + (rest + wrows - 1) / wrows;
  if (ks == 1) planned_us = rounds_us(shape, M, columns, N, K, 0);   // (the plan of one product knows no sections)
  return us < 0.98 * planned_us ? tile : 0;
}

// shape: 0: chosen here; else stages * 1000000 + rows * 1000 + weight rows of a workgroup's tile (2256192, 3256128,
// 3128256, 3192128; 2128192: workgroups of four waves, two to a CU).
// ks > 1 cuts K over that many workgroups per tile (no epilogue only; the partial tiles go through `workspace`,
// which must hold ks * M * N floats).
int gemm_wide(const void* A, int64_t lda, const void* W, void* C, int64_t ldc, int M, int N, int K, int epi, int act,
              float limit, int shape, int ks, void* workspace, size_t workspace_bytes, hipStream_t stream, int* planes_left, int c_dtype,
              Sections sec) {
  if (ks < 1) ks = 1;
  if (ks > K / wide::BK) ks = K / wide::BK;
  if (ks > 1 && (epi != 0 || workspace == nullptr || static_cast<size_t>(ks) * M * N * sizeof(float) > workspace_bytes)) {
    set_error("gemm: the wide kernel cuts K only without an epilogue and with a workspace of ks * M * N floats");
    return 1;
  }
  float* ws = static_cast<float*>(workspace);
  const bf16* a = static_cast<const bf16*>(A);
  const bf16* w = static_cast<const bf16*>(W);
  bf16* c = static_cast<bf16*>(C);
  // (the broad kernel stores pieces of eight columns)
  const bool broad = N % 8 == 0 && ldc % 8 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
  const bool planned = shape == 0;
  double planned_us = 0.0;
  if (planned) planned_us = plan_shape(M, N, K, epi, ws != nullptr, workspace_bytes, shape, ks, planes_left != nullptr, broad && sec.n_step == 0);
  if (shape / 1000000 == 1 && !broad) {
    set_error("gemm: the broad tiles want widths and rows of whole pieces of eight columns");
    return 1;
  }
  // Several products at once: where the broad kernel's tiles are ahead, the whole sections run on it and a shorter last one by itself.
  const int broad_tile = planned && broad && c_dtype == kBF16 ? sections_broad_tile(M, N, K, sec.n_step, ws != nullptr, workspace_bytes, shape, ks, planned_us) : 0;
  if (broad_tile > 0) {
    const int whole = N / sec.n_step, rest = N % sec.n_step;
    gemm_broad(broad_tile, a, lda, w, c, ldc, M, whole * sec.n_step, K, 0, 0, 0.f, 1, nullptr, false, sec, stream);
    if (check_launch("gemm_broad")) return 1;
    const size_t at = static_cast<size_t>(whole) * sec.n_step;
    return rest == 0 ? 0 : sa_gemm(a + static_cast<size_t>(whole) * sec.a_step, kBF16, lda, w + at * K, nullptr, kBF16, c + at, kBF16, ldc,
                                   M, rest, K, 0, 0.f, 0, 1, 0, workspace, static_cast<int64_t>(workspace_bytes), stream);
  }
  // 32-bit results: the cuts' partial sums as they are, of one cut straight into C (whose rows are contiguous)
  const bool raw = ks > 1 || c_dtype == kF32;
  float* to = ks > 1 ? ws : static_cast<float*>(C);
  switch (shape) {
    case 2256192: wide::launch<4, 6, 4, 2>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 3256128: wide::launch<4, 4, 4, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 3128256: wide::launch<4, 4, 2, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 3192128: wide::launch<3, 4, 4, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 2128192: wide::launch<4, 6, 2, 2, 4>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;  // two workgroups per CU
    // small tiles, for products of a few hundred rows whose large tiles would leave most CUs idle (two or more
    // workgroups per CU fit: 36 to 72 KiB of LDS each)
    case 3128128: wide::launch<2, 4, 4, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 3128064: wide::launch<2, 2, 4, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 3064128: wide::launch<1, 4, 4, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 3064064: wide::launch<1, 2, 4, 3>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 6064064: wide::launch<1, 2, 4, 6>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 5128064: wide::launch<2, 2, 4, 5>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 4128128: wide::launch<2, 4, 4, 4>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    case 1256256: case 1256288: case 1192256: case 1192288:
      gemm_broad(shape % 1000000, a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream);
      break;
    case 6064128: wide::launch<1, 4, 4, 6>(a, lda, w, c, ldc, M, N, K, epi, act, limit, ks, to, raw, sec, stream); break;
    default:
      set_error("gemm: unknown wide tile %d", shape);
      return 1;
  }
  if (check_launch("gemm_wide")) return 1;
  if (planes_left != nullptr) {  // the caller adds the cuts' partial results up itself (ks planes of [M, N] floats)
    *planes_left = ks;
    return 0;
  }
  if (ks > 1) {
    if (gemm_sum_partials(ws, ks, C, c_dtype, ldc, M, N, N, 0, 0, 0.f, stream)) return 1;
    if (epi == 0 && act > 0) return apply_activation(C, kBF16, ldc, M, N, act - 1, stream);   // (the kernels with K cut have no such epilogue)
  }
  return 0;
}


double gemm_wide_predict_us(int M, int N, int K, int epi, bool have_workspace, size_t workspace_bytes, bool planes) {
  int shape = 0, ks = 1;
  return plan_shape(M, N, K, epi, have_workspace, workspace_bytes, shape, ks, planes);
}

}  // namespace sa

extern "C" int sa_gemm_wide_shape(int M, int N, int K, int epilogue, int64_t workspace_bytes) {
  if (M < 1 || N < 1 || K < 1 || epilogue < 0 || epilogue > 1) return 0;
  int shape = 0, ks = 1;
  const size_t bytes = workspace_bytes > 0 ? static_cast<size_t>(workspace_bytes) : 0;
  sa::plan_shape(M, N, K, epilogue, bytes > 0, bytes, shape, ks, false, false);
  return shape;
}

static int broad_tile(int M, int N, int K, int epi, int64_t workspace_bytes, bool planes) {
  if (M < 1 || N < 1 || K < 1 || epi < 0 || epi > 1) return 0;
  int shape = 0, ks = 1;
  const size_t bytes = workspace_bytes > 0 ? static_cast<size_t>(workspace_bytes) : 0;
  sa::plan_shape(M, N, K, epi, bytes > 0, bytes, shape, ks, planes);
  return shape / 1000000 == 1 ? (ks - 1) * 1000000 + shape : 0;
}

extern "C" int sa_gemm_broad_tile(int M, int N, int K, int epilogue, int64_t workspace_bytes) {
  return broad_tile(M, N, K, epilogue, workspace_bytes, false);
}

extern "C" int sa_gemm_planes_broad_tile(int M, int N, int K, int64_t workspace_bytes) {
  return broad_tile(M, N, K, 0, workspace_bytes, true);
}

extern "C" int sa_gemm_sections_tile(int M, int N, int K, int n_step, int64_t workspace_bytes) {
  if (M < 1 || N < 1 || K < 1 || n_step < 1) return 0;
  int shape = 0, ks = 1;
  const size_t bytes = workspace_bytes > 0 ? static_cast<size_t>(workspace_bytes) : 0;
  const double us = sa::plan_shape(M, N, K, 0, bytes > 0, bytes, shape, ks, false, false);
  return sa::sections_broad_tile(M, N, K, n_step, bytes > 0, bytes, shape, ks, us);
}
