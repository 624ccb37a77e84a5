// Paged attention in bfloat16 for prompts whose many query heads share one long key vector (latents: keys of a latent and
// a rotated part, values of the latent alone).  attention_maps.hip takes one unit of 16 query rows to a workgroup and
// reads all of the keys and values for it: with 1,088 entries a key that is the bound (16 heads and one token a unit,
// the L2 caches).  Here a workgroup of eight waves takes a group of four units of one request, and the keys and values
// of a tile of 32 keys come into LDS once for all of its 64 rows.
//
// Two waves go with a unit.  Per tile
//     S^T = K . Q^T         each of the two takes half of the tile's keys, the unit's queries in registers
//     mask and row maxima   of the halves, exchanged through LDS
//     online softmax        in float32 (base-2 exponentials); P^T and the rows' rescaling factors go to LDS
//     O^T += V^T . P^T      all four units, the wave's own eighth of the value entries: a value block is read once
// The exchange of P^T costs 4 KiB of LDS a tile and saves reading the values four times.  The second product of a tile
// follows in the next step, among the scores of the next tile, whose operands it covers, and the last four of it cover
// the exchange of the maxima; a step has two barriers, of which the first publishes P^T of the tile before and the loads
// that were asked for during the step before.  Keys and values are both kept in two buffers, 2 * (32 * 1,088) * 2 bytes in all for
// the largest sizes, so one workgroup of eight waves runs on a CU.
// (Four waves with a SIMD each and twice the accumulators needed more than 256 registers; the compiler then moved all
// accumulators between the halves of the register file in every step, for the sake of the rare rescaling: 184 us.)
//
// Measured, 16 heads over one key of 576 entries and values of 512: a prompt of 2,047 tokens 553 -> 132 us, of 4,095
// 2,371 -> 436, of 512 90 -> 49; 64 tokens behind 8,000 213 -> 51; keys of 192 and values of 128, 1,000 tokens 70 -> 46
// (of which the look for values that are not finite, in tiles that not every unit sees whole, is 1 to 2 %).
// Without the loads (in a copy) 2,047 tokens took 95 us: LDS is the bound, 208 KiB through it per tile, with the chain
// score - maximum - exchange - exponential behind it; with the second product after the maxima instead of among the
// scores it was 135.
#include "api.h"
#include "attention_common.h"

namespace sa {
namespace groups {

constexpr int kUnits = 4;    // units per workgroup
constexpr int kWaves = 8;    // two per unit
constexpr float kLog2e = 1.4426950408889634f;

// Every load into LDS has arrived and every LDS access is done, then the workgroup barrier.  The empty statements and the
// scheduling barriers keep the compiler from moving memory accesses across it (it does not know of the loads into LDS).
__device__ inline void publish() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((7 << 4));   // vmcnt(0) lgkmcnt(0), expcnt left alone
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

// The barrier alone, behind this wave's LDS accesses; loads may be under way.
__device__ inline void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((7 << 4) | 15 | (3 << 14));   // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

struct Shape {
  int Kh, chunks, Gc, G_all;   // key heads; chunks of Gc query heads per key head (G_all in all)
  int page_size, window, chunk_tiles;
  float scale2;                // the scores' factor times log2(e)
};

// NDC: 32-entry blocks of a key vector.  VPW: 16-entry blocks of values that a wave owns.
template <int NDC, int VPW>
__global__ __launch_bounds__(kWaves * kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) void paged_attention_groups_kernel(
    const bf16* __restrict__ q, int64_t q_stride, const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const SeqMeta* __restrict__ units, int unit_begin,
    bf16* __restrict__ out, int64_t out_stride, Shape sh, float* __restrict__ workspace) {
  constexpr int HD = NDC * 32, NDB = VPW * kWaves, HDV = NDB * 16;
  constexpr int K_BLOCKS = 2 * NDC;                         // KiB of keys per tile
  constexpr int KPW = (K_BLOCKS + kWaves - 1) / kWaves;     // of them asked for by a wave
  __shared__ __attribute__((aligned(16))) __bf16 k_stage[2][K_BLOCKS * 512];
  __shared__ __attribute__((aligned(16))) __bf16 v_stage[2][NDB * 512];
  __shared__ __attribute__((aligned(16))) bf16x8 p_s[2][kUnits][kWave];
  __shared__ float alpha_s[2][kUnits * 16];
  __shared__ float max_s[2][kWaves * 16];
  const uint32_t k_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) __bf16*)&k_stage[0][0])) ;
  const uint32_t v_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) __bf16*)&v_stage[0][0])) ;

  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t k_lds = k_at + wave * 1024, v_lds = v_at + wave * 1024;
  const int u = wave % kUnits, half = wave / kUnits;   // the wave's unit, and its half of a tile's keys
  const int r = lane % 16, grp = lane / 16;
  const int split = blockIdx.y, num_splits = gridDim.y, vy = blockIdx.x, KhV = gridDim.x;
  const int kh = vy / sh.chunks, chunk = vy % sh.chunks;
  // later units of a prompt see more keys: they are started first
  const int group = gridDim.z - 1 - blockIdx.z;
  const int u0 = unit_begin + group * kUnits;
  const int Gc = sh.Gc, page_size = sh.page_size, window = sh.window;

  int lo_g, hi_g, slot = 0;
  if (!group_keys(units, u0, kUnits, window, &lo_g, &hi_g, &slot)) return;   // no rows at all
  lo_g = __builtin_amdgcn_readfirstlane(lo_g), hi_g = __builtin_amdgcn_readfirstlane(hi_g);
  // where the first unit's keys end and where the last one's begin: every unit sees the keys between whole
  int hi_first = hi_g, lo_last_unit = lo_g;
  for (int w = 0; w < kUnits; ++w) {
    const SeqMeta m = units[u0 + w];
    if (m.q_len <= 0) continue;
    hi_first = min(hi_first, m.pos0 + m.q_len);
    if (window > 0) lo_last_unit = max(lo_last_unit, m.pos0 - window + 1);
  }
  hi_first = __builtin_amdgcn_readfirstlane(hi_first), lo_last_unit = __builtin_amdgcn_readfirstlane(lo_last_unit);
  const int tile0 = lo_g / kTile, tile1 = (hi_g + kTile - 1) / kTile;
  const int num_chunks = key_chunks(lo_g, hi_g, sh.chunk_tiles);
  if (split >= num_chunks) return;   // (the same for the whole workgroup)
  const int* table = block_table + static_cast<size_t>(__builtin_amdgcn_readfirstlane(slot)) * table_stride;
  const int tb = tile0 + split * sh.chunk_tiles;
  const int te = tb + sh.chunk_tiles < tile1 ? tb + sh.chunk_tiles : tile1;

  // the unit of this wave, this lane's row of it (query token qi, query head g of the chunk) and its queries as B operands:
  // lane (row r, grp) holds Q[row r][dc * 32 + grp * 8 .. + 8]
  const int qi = r / Gc, g = r % Gc;
  const SeqMeta sm = units[u0 + u];
  const int rows = Gc * sm.q_len;   // <= 16
  const bool row_ok = r < rows;
  const int pos_r = sm.pos0 + qi;
  const int lo_r = (window > 0 && pos_r - window + 1 > 0) ? pos_r - window + 1 : 0;
  const int pos_last = sm.pos0 + sm.q_len - 1;
  const int lo_last = (window > 0 && pos_last - window + 1 > 0) ? pos_last - window + 1 : 0;
  bf16x8 qf[NDC];
  {
    const bf16* qp = q + static_cast<size_t>(row_ok ? sm.q_start + qi : units[u0].q_start) * q_stride +
                     static_cast<size_t>(kh * sh.G_all + chunk * Gc + (row_ok ? g : 0)) * HD + grp * 8;
#pragma unroll
    for (int dc = 0; dc < NDC; ++dc) qf[dc] = row_ok ? *reinterpret_cast<const bf16x8*>(qp + dc * 32) : bf16x8{};
  }
  floatx4 acc[kUnits][VPW];   // O^T of unit w, value entries (wave * VPW + j) * 16 + 4 * grp + v, row r
#pragma unroll
  for (int w = 0; w < kUnits; ++w)
#pragma unroll
    for (int j = 0; j < VPW; ++j) acc[w][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;   // of this wave's unit; l_run is this wave's and lane group's share

  // How a tile lies in LDS: product t of the scores takes, as row i of its A operand, key 8 * (i / 4) + 4 * t + i % 4
  // of the tile, so that a lane's scores of both belong to the keys 8 * grp .. + 7 and are the second product's operand
  // as they stand; a wave computes product t = half.  Blocks of 64 lanes x 16 bytes in the order of the lanes that read them; the load into LDS picks the
  // matching 16 bytes of the pages.
  //   key block 2 dc + t, lane (kgrp, i):  sub-tile i / 8 of the tile, its key 8 * ((i / 4) % 2) + 4 * t + i % 4
  //   value block db, lane (grp, r):       sub-tile grp / 2, keys 8 * (grp % 2) .. + 7 of entry 16 * db + r
  const int row = lane % 16;
  const int k_sub = row / 8, v_sub = lane / 32;   // the sub-tile that this lane's pieces come from
  // (a wave asks for blocks wave, wave + 8, ...: always the same t, and steps of constant size through the pages)
  const uint32_t k_lane = ((lane / 16) * 16 + 8 * ((row / 4) % 2) + row % 4 + (wave % 2) * 4) * 8 + (wave / 2) * 512;
  const uint32_t v_lane = (wave * 16 + row) * page_size + ((lane / 16) % 2) * 8;
  const uint32_t v_step = kWaves * 16 * page_size;
  int blk[2], off[2];   // block of the table and key of its page of the two sub-tiles that are looked up next
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int sk0 = tb * kTile + n * 16;
    blk[n] = __builtin_amdgcn_readfirstlane(sk0 / page_size);
    off[n] = __builtin_amdgcn_readfirstlane(sk0 % page_size);
  }
  // the blocks of the table that this workgroup's keys lie in
  const int blk_lo = lo_g / page_size, blk_hi = (min(hi_g, te * kTile) - 1) / page_size;
  struct Pages {
    uint32_t page[2], at[2];
  };
  // (called for consecutive tiles; a sub-tile outside of the keys reads the nearest page, and what it brings is dropped)
  auto look_up = [&]() __attribute__((always_inline)) {
    Pages p;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      p.page[n] = static_cast<uint32_t>(table[min(max(blk[n], blk_lo), blk_hi)]);
      p.at[n] = static_cast<uint32_t>(off[n]);
      off[n] += kTile;
#pragma unroll
      for (int twice = 0; twice < 2; ++twice)
        if (off[n] >= page_size) {
          off[n] -= page_size;
          ++blk[n];
        }
    }
    return p;
  };
  const uint32_t k_page = static_cast<uint32_t>(sh.Kh) * page_size * HD, v_page = static_cast<uint32_t>(sh.Kh) * page_size * HDV;
  const bf16* const k_head = k_pages + static_cast<int64_t>(kh) * page_size * HD + k_lane;
  const bf16* const v_head = v_pages + static_cast<int64_t>(kh) * page_size * HDV + v_lane;
  auto keys_at = [&](const Pages& p) __attribute__((always_inline)) {
    const uint32_t page = k_sub ? p.page[1] : p.page[0], at = k_sub ? p.at[1] : p.at[0];
    return k_head + static_cast<uint64_t>(page) * k_page + (at >> 4) * (NDC * 512);
  };
  auto values_at = [&](const Pages& p) __attribute__((always_inline)) {
    const uint32_t page = v_sub ? p.page[1] : p.page[0], at = v_sub ? p.at[1] : p.at[0];
    return v_head + static_cast<uint64_t>(page) * v_page + at;
  };
  auto ask_keys = [&](int i, const bf16* from, uint32_t to) __attribute__((always_inline)) {
    if (K_BLOCKS % kWaves != 0 && i == KPW - 1 && wave + kWaves * i >= K_BLOCKS) return;
    __builtin_amdgcn_sched_barrier(0);
    load_to_lds(from + i * (kWaves * 256), to + i * (kWaves * 1024));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto ask_values = [&](int i, const bf16*& from, uint32_t to) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    load_to_lds(from, to + i * (kWaves * 1024));
    from += v_step;
    __builtin_amdgcn_sched_barrier(0);
  };

  // O^T += V^T . P^T of tile `tile`, which lies in the buffers `b`
  bf16x8 vf[VPW], pf[kUnits];
  float alpha[kUnits];
  auto read_second = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < kUnits; ++w) {
      pf[w] = p_s[b][w][lane];
      alpha[w] = alpha_s[b][w * 16 + r];
    }
#pragma unroll
    for (int j = 0; j < VPW; ++j)
      vf[j] = *reinterpret_cast<const bf16x8*>(&v_stage[b][0] + wave * VPW * 512 + lane * 8 + j * 512);
  };
  auto rescale_second = [&](int tile) __attribute__((always_inline)) {
    bool any = false;
#pragma unroll
    for (int w = 0; w < kUnits; ++w) any = any || alpha[w] != 1.f;
    if (__builtin_amdgcn_ballot_w64(any) != 0) {   // rarely, once the maxima have settled
#pragma unroll
      for (int w = 0; w < kUnits; ++w)
#pragma unroll
        for (int j = 0; j < VPW; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[w][j][v] *= alpha[w];
    }
    const int key0 = tile * kTile;
    if (__builtin_expect(key0 + kTile <= hi_first && key0 >= lo_last_unit, 1)) return;
    // keys that no row may use (unwritten, given back) count as 0
    constexpr uint32_t kExponents = 0x7f807f80u;
    typedef __attribute__((ext_vector_type(4))) uint32_t Pairs;   // of neighbouring keys
    auto between = [&](int lo, int hi) __attribute__((always_inline)) {
      Pairs m;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key0 + grp * 8 + 2 * i;
        m[i] = (key >= lo && key < hi ? 0xffffu : 0u) | (key + 1 >= lo && key + 1 < hi ? 0xffff0000u : 0u);
      }
      return m;
    };
    const Pairs used = between(lo_g, hi_g);
    bool odd = false;
#pragma unroll
    for (int j = 0; j < VPW; ++j) {
      const Pairs v = __builtin_bit_cast(Pairs, vf[j]) & used;
      vf[j] = __builtin_bit_cast(bf16x8, v);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t e = v[i] & kExponents;
        odd |= (e & 0xffffu) == (kExponents & 0xffffu) || e >> 16 == kExponents >> 16;
      }
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd) == 0, 1)) return;
    // Keys that some units see and others do not, with values that are not finite, which a probability of zero does not
    // take out: each unit's products here, without the keys that it does not see, and none later.
#pragma unroll
    for (int w = 0; w < kUnits; ++w) {
      const SeqMeta m = units[u0 + w];
      const Pairs seen = between(window > 0 ? m.pos0 - window + 1 : 0, m.pos0 + m.q_len);
#pragma unroll
      for (int j = 0; j < VPW; ++j)
        acc[w][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, __builtin_bit_cast(Pairs, vf[j]) & seen),
                                                            pf[w], acc[w][j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < VPW; ++j) vf[j] = bf16x8{};
  };
  auto second = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
    for (int j = from; j < to; ++j)
#pragma unroll
      for (int w = 0; w < kUnits; ++w)
        acc[w][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[j], pf[w], acc[w][j], 0, 0, 0);
  };

  Pages here, next;   // of the tile whose keys have been asked for, and of the one after it
  // scores of `tile` from key buffer b, the second product of the tile before from the other buffers; meanwhile the
  // keys of the next tile and the values of this one are asked for
  auto step = [&](int tile, int b, bool first) __attribute__((always_inline)) {
    const bf16* k_from = keys_at(next);
    const bf16* v_from = values_at(here);
    const uint32_t k_to = k_lds + (b ^ 1) * (K_BLOCKS * 1024), v_to = v_lds + b * (NDB * 1024);
    constexpr int KB = 3, KBATCHES = (NDC + KB - 1) / KB;
    floatx4 s2[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};   // (two chains of products)
    bf16x8 kf[2][KB];
    const __bf16* k_mine = &k_stage[b][0] + half * 512 + lane * 8;
    auto read_keys = [&](int batch) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < KB; ++i)
        if (batch * KB + i < NDC)
          kf[batch % 2][i] = *reinterpret_cast<const bf16x8*>(k_mine + (batch * KB + i) * 1024);
    };
    if (!first) read_second(b ^ 1);
    read_keys(0);
    if (!first) rescale_second(tile - 1);
#pragma unroll
    for (int batch = 0; batch < KBATCHES; ++batch) {
      if (batch + 1 < KBATCHES) read_keys(batch + 1);
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int dc = batch * KB + i;
        if (dc >= NDC) break;
        s2[dc % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[batch % 2][i], qf[dc], s2[dc % 2], 0, 0, 0);
        // among the scores' products those of the tile before (but for the last four), and the loads, asked for one by one
        if (!first && dc < 4 * (VPW - 1))
          acc[dc % 4][dc / 4] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dc / 4], pf[dc % 4], acc[dc % 4][dc / 4], 0, 0, 0);
        if (dc % 2 == 0) {
          if (dc / 2 < KPW) ask_keys(dc / 2, k_from, k_to);
        } else if (dc / 2 < VPW) {
          ask_values(dc / 2, v_from, v_to);
        }
      }
    }
    static_assert(KPW <= (NDC + 1) / 2 && VPW <= NDC / 2 && kUnits * (VPW - 1) <= NDC, "what goes among the scores");
    const int key0 = tile * kTile;
    float y[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) y[v] = (s2[0][v] + s2[1][v]) * sh.scale2;
    if (!(rows == 16 && key0 + kTile - 1 <= sm.pos0 && key0 >= lo_last)) {   // (uniform: some row does not see it whole)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int key = key0 + grp * 8 + half * 4 + v;
        y[v] = (row_ok && key <= pos_r && key >= lo_r) ? y[v] : -INFINITY;
      }
    }
    const float mine = max_over_row_lanes(fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3])));
    if (grp == 0) max_s[b][wave * 16 + r] = mine;
    // (the table's entries arrive during the rest of the products: a wait for LDS is a wait for scalar loads as well)
    __builtin_amdgcn_sched_barrier(0);
    here = next;
    next = look_up();
    __builtin_amdgcn_sched_barrier(0);
    if (!first) second(VPW - 1, VPW);
    meet();
    const float m_new = fmaxf(m_run, fmaxf(mine, max_s[b][(wave ^ kUnits) * 16 + r]));
    // a row that has seen no visible key yet keeps m = -inf; 2^(-inf - -inf) must not appear
    const float factor = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    float psum = 0.f;
    bf16x4 p;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float e = __builtin_amdgcn_exp2f(y[v] - m_use);   // 2^-inf = 0
      psum += e;
      p[v] = to_bf16_raw(e);
    }
    l_run = l_run * factor + psum;
    m_run = m_new;
    reinterpret_cast<bf16x4*>(&p_s[b][u][lane])[half] = p;
    if (half == 0 && grp == 0) alpha_s[b][u * 16 + r] = factor;
  };

  // (te > tb: every range below num_chunks has a tile)
  here = look_up();
  next = look_up();
  {
    const bf16* k_from = keys_at(here);
#pragma unroll
    for (int i = 0; i < KPW; ++i) ask_keys(i, k_from, k_lds);
  }
  publish();
  step(tb, 0, true);
  int b = 1;
#pragma unroll 1
  for (int tile = tb + 1; tile < te; ++tile, b ^= 1) {
    publish();
    step(tile, b, false);
  }
  publish();
  {
    read_second(b ^ 1);
    rescale_second(te - 1);
    second(0, VPW);
  }
  // the rows' sums of both halves: every wave needs those of all units
  float* sums = &max_s[b][0];   // (not the buffer that the last step has read)
  const float l = sum_over_row_lanes(l_run);
  if (grp == 0) sums[wave * 16 + r] = l;
  publish();
  const int unit_of_group = group * kUnits;
#pragma unroll
  for (int w = 0; w < kUnits; ++w) {
    const SeqMeta um = units[u0 + w];
    if (r >= Gc * um.q_len) continue;
    if (num_chunks == 1) {
      bf16* op = out + static_cast<size_t>(um.q_start + qi) * out_stride + static_cast<size_t>(vy * Gc + g) * HDV;
      const float inv = 1.f / (sums[w * 16 + r] + sums[(w + kUnits) * 16 + r]);
#pragma unroll
      for (int j = 0; j < VPW; ++j) {
        const bf16x4 o4 = {to_bf16_raw(acc[w][j][0] * inv), to_bf16_raw(acc[w][j][1] * inv),
                           to_bf16_raw(acc[w][j][2] * inv), to_bf16_raw(acc[w][j][3] * inv)};
        *reinterpret_cast<bf16x4*>(op + (wave * VPW + j) * 16 + 4 * grp) = o4;
      }
    } else {
      float* wp = workspace +
                  ((static_cast<size_t>(unit_of_group + w) * KhV + vy) * num_splits + split) * 16 * (HDV + kRowExtra) +
                  r * (HDV + kRowExtra);
#pragma unroll
      for (int j = 0; j < VPW; ++j) *reinterpret_cast<floatx4*>(wp + (wave * VPW + j) * 16 + 4 * grp) = acc[w][j];
    }
  }
  if (num_chunks > 1 && half == 0 && grp == 0 && row_ok) {   // (the merge kernel works with natural logarithms)
    float* wp = workspace +
                ((static_cast<size_t>(unit_of_group + u) * KhV + vy) * num_splits + split) * 16 * (HDV + kRowExtra) +
                r * (HDV + kRowExtra) + HDV;
    wp[0] = m_run * (1.f / kLog2e);
    wp[1] = l + sums[(wave + kUnits) * 16 + r];
  }
}

}  // namespace groups

}  // namespace sa

using namespace sa;

extern "C" int sa_paged_attention_groups_size() { return groups::kUnits; }

// The tiles of 32 keys that a unit of such a launch sees on average: a fresh prompt's units see half of its keys, those
// of a portion behind many keys all of them.
static int average_tiles(int unit_count, int window, int max_kv_len, int max_q_len) {
  const int64_t span = window > 0 && window < max_kv_len ? window + 16 * groups::kUnits : max_kv_len;
  const int64_t tokens = static_cast<int64_t>(unit_count) * max_q_len;
  return static_cast<int>((span - (tokens < span ? tokens : span) / 2) / kTile + 1);
}

// Whether sa_paged_attention_groups takes these sizes: values of 128, 256 or 512 entries, keys of as many or 32 or 64
// more, and what sa_paged_attention_maps_units asks of pages and alignments.
extern "C" int sa_paged_attention_groups_takes(int H, int Kh, int hd, int hd_v, int page_size, int64_t q_stride,
                                               const void* q) {
  return (hd_v == 128 || hd_v == 256 || hd_v == 512) && (hd == hd_v || hd == hd_v + 32 || hd == hd_v + 64) &&
         sa_paged_attention_maps_units_takes(H, Kh, 1, hd, hd_v, page_size, q_stride, q);
}

// Whether so many units are better taken in groups: from about 640 pairs of a unit and a tile of keys.  Values of 512:
// 8 tokens behind 3,000 keys took 23.0 us unit by unit and 22.3 in groups, 16 behind 1,000 19.5 and 21.3, 64 of 8
// requests behind 300 22.9 and 23.8, 32 behind 1,000 27.8 and 23.7.
extern "C" int sa_paged_attention_groups_pays(int unit_count, int H, int Kh, int window, int max_kv_len, int max_q_len) {
  const int Gc = H > 0 && Kh > 0 && H % Kh == 0 ? sa_attention_maps_heads_per_unit(H, Kh) : 1;
  return static_cast<int64_t>(unit_count) * (H / Gc) * average_tiles(unit_count, window, max_kv_len, max_q_len) >= 640;
}

// What sa_paged_attention_maps_units computes with one map, over units whose consecutive groups of
// sa_paged_attention_groups_size() belong to one request each (empty units where its tokens end).
extern "C" int sa_paged_attention_groups(const void* q, int64_t q_stride, const void* k_pages, const void* v_pages,
                                         const int* block_table, int table_stride, const int* units, int unit_begin,
                                         int unit_count, void* out, int64_t out_stride, int H, int Kh, int hd, int hd_v,
                                         int page_size, int window, float scale, int max_kv_len, int max_q_len,
                                         void* workspace, size_t workspace_bytes, hipStream_t stream) {
  constexpr int kGroup = groups::kUnits;
  if (unit_count == 0) return 0;
  SA_REQUIRE(unit_count > 0 && unit_begin >= 0 && table_stride > 0 && window >= 0 && max_kv_len > 0 && max_q_len > 0,
             "paged_attention_groups: bad counts, window, table or lengths");
  SA_REQUIRE(unit_count % kGroup == 0, "paged_attention_groups: %d units are no whole groups of %d", unit_count, kGroup);
  SA_REQUIRE(sa_paged_attention_groups_takes(H, Kh, hd, hd_v, page_size, q_stride, q),
             "paged_attention_groups takes values of 128, 256 or 512 entries, keys of up to 64 more, pages of a multiple "
             "of 16 keys and aligned query rows; got hd=%d hd_v=%d P=%d", hd, hd_v, page_size);
  SA_REQUIRE(q_stride >= static_cast<int64_t>(H) * hd && out_stride >= static_cast<int64_t>(H) * hd_v,
             "paged_attention_groups: row strides are below what the heads need");
  SA_REQUIRE(out_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
             "paged_attention_groups: output rows are aligned to 8 bytes");
  const int G = H / Kh, Gc = sa_attention_maps_heads_per_unit(H, Kh);
  SA_REQUIRE(Gc * max_q_len <= 16, "paged_attention_groups: units of %d tokens x %d heads exceed 16 rows", max_q_len, Gc);
  groups::Shape sh;
  sh.Kh = Kh, sh.chunks = G / Gc, sh.Gc = Gc, sh.G_all = G;
  sh.page_size = page_size, sh.window = window, sh.scale2 = scale * groups::kLog2e;
  const int KhV = Kh * sh.chunks, count = unit_count / kGroup;
  SA_REQUIRE(count <= 65535, "paged_attention_groups: too many units");
  // Ranges of keys: as many as bring one workgroup to a CU, of 4 tiles at least, or of 8 that read fewer
  // entries (a range costs its set-up and the partial results' way through memory). 
  const int span = window > 0 && window < max_kv_len ? window + 16 * kGroup : max_kv_len;
  const int max_tiles = (span + kTile - 1) / kTile + 1;
  const int64_t avg_tiles = average_tiles(unit_count, window, max_kv_len, max_q_len);
  int64_t ranges = 256 * static_cast<int64_t>(max_tiles) / (static_cast<int64_t>(count) * KhV * avg_tiles);
  const int least = hd_v > 256 ? 4 : 8;
  if (ranges > max_tiles / least) ranges = max_tiles / least;
  if (ranges < 1) ranges = 1;
  int chunk = static_cast<int>((max_tiles + ranges - 1) / ranges);
  int KS = (max_tiles + chunk - 1) / chunk;
  const size_t per_split = static_cast<size_t>(unit_count) * KhV * 16 * (hd_v + kRowExtra) * sizeof(float);
  while (KS > 1 && (KS > kMaxSplits || workspace == nullptr || per_split * KS > workspace_bytes)) {
    ++chunk;
    KS = (max_tiles + chunk - 1) / chunk;
  }
  sh.chunk_tiles = chunk;
  const dim3 grid(KhV, KS, count);
  const bf16* qp = static_cast<const bf16*>(q);
  const bf16* kp = static_cast<const bf16*>(k_pages);
  const bf16* vp = static_cast<const bf16*>(v_pages);
  const SeqMeta* um = reinterpret_cast<const SeqMeta*>(units);
  bf16* op = static_cast<bf16*>(out);
  float* ws = static_cast<float*>(workspace);
#define SA_LAUNCH(NDC, VPW)                                                                                             \
  groups::paged_attention_groups_kernel<NDC, VPW><<<grid, groups::kWaves * kWave, 0, stream>>>(qp, q_stride, kp, vp, block_table,          \
                                                                            table_stride, um, unit_begin, op, out_stride, \
                                                                            sh, ws)
  const int more = (hd - hd_v) / 32;
  if (hd_v == 128) {
    if (more == 0) SA_LAUNCH(4, 1);
    else if (more == 1) SA_LAUNCH(5, 1);
    else SA_LAUNCH(6, 1);
  } else if (hd_v == 256) {
    if (more == 0) SA_LAUNCH(8, 2);
    else if (more == 1) SA_LAUNCH(9, 2);
    else SA_LAUNCH(10, 2);
  } else {
    if (more == 0) SA_LAUNCH(16, 4);
    else if (more == 1) SA_LAUNCH(17, 4);
    else SA_LAUNCH(18, 4);
  }
#undef SA_LAUNCH
  if (check_launch("paged_attention_groups")) return 1;
  if (KS > 1)
    return attention_merge_ranges(ws, KS, hd_v, um, unit_begin, unit_count, max_q_len, op, out_stride, KhV, Gc, stream,
                                  chunk, kGroup, window, nullptr);
  return 0;
}
