#pragma once
// Prefill chunk rows on MFMA, 16-bit caches (hot-path part 3): the prefill
// tile's workgroup.
//
// The same function as the chunk tile (attention_chunk_wg.h) with a 16-bit
// cache, for every step that gives no tile or partition size (cut_prefill in
// step_plan.cpp). The chunk tile is bound by LDS reads (each wave reads a K/V
// tile for its 32 rows of one head: 8 waves read 128 KB of LDS per 64 keys),
// by idle waves (one wave per query head of the group: half of them with
// G = 4, seven of eight with G = 1), by a load phase that nothing overlaps,
// and by the partials of its 384-key partitions. Measured, chunk tile against
// this one (us; the kernel alone, back to back, untraced: a profiler's launches
// run up to 10 % longer): 4096 rows after 0-1536 keys, 32/4
// heads x 64, 131 against 63 (706 TFLOP/s); 2048 rows after 8192, 32/8 x 128,
// 845 against 357 (865); 4096 rows after 4096, 32/4 x 64, 369 against 164
// (890); 512 rows after 1024, 14/2 x 64, 18.5 against 15.4; 4 x 512 rows after
// 4096, 8/8 x 128, 419 against 69. What bounds it now: with the chip full, the
// matrix cores' issue beside the softmax's vector work on the same SIMDs
// (counters of the 2048 rows after 8192: MFMA busy 36 % of a SIMD's cycles,
// vector instructions active 45 %, LDS 36 %; a large bf16 GEMM reaches 1200-1370
// TFLOP/s on this card); in small steps the
// serial chain of a tile (fragments, product, max, exp2, product, barrier:
// about 1 us per 64 keys with one workgroup on a CU).
//
// gfx950 design:
//   * a workgroup owns 128 (wide: 256) query columns of one kv head, column
//     c = (row c / G, head c % G) of consecutive rows, so every wave is busy
//     whatever the group; a wave owns 32 (64) columns as NC = 1 (2) column
//     tiles that share every K and V fragment read from LDS;
//   * four waves and 64-key tiles, double buffered in LDS (one barrier a
//     tile), the following tiles' global loads in flight in registers during
//     a tile's products. Two workgroups share a CU (at most 256 VGPRs), so
//     one's softmax runs beside the other's MFMAs;
//   * S^T = K . Q^T and O^T = V^T . P^T on the 32x32x16 MFMA: a lane holds one
//     query column, its P^T accumulators are the B operand of the second
//     product as they are (A and B only have to agree on the key order), V^T
//     comes from row-major V rows through ds_read_b64_tr_b16;
//   * softmax: a score leaves the MFMA less its column's base (the C operand),
//     so a tile's vector work per score is max, exp2, a packed conversion and a
//     two-wide dot with ones for the row sum; the base is the maximum of the
//     column's first tile and moves when scores pass it by more than 8 (log2).
#include <float.h>

#include "attention_chunk_wg.h"

namespace le {
namespace pre {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWave;
constexpr int kTileKeys = 64;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <typename T> struct mma32;
template <> struct mma32<bf16_t> {
  using v2 = bf16x2;
  __device__ __forceinline__ static f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static float dot2(v2 a, v2 b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(a, b, c, false);
  }
};
template <> struct mma32<f16_t> {
  using v2 = f16x2;
  __device__ __forceinline__ static f32x16 mma(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static float dot2(v2 a, v2 b, float c) { return __builtin_amdgcn_fdot2(a, b, c, false); }
};

// K rows are padded by 16 bytes (the 16-byte fragment reads of 8 consecutive
// rows then cover all banks), V rows by 32 (the transposing reads of 4 rows x
// 32 bytes do).
template <int HD> struct Lds {
  static constexpr int KROW = HD * 2 + 16, VROW = HD * 2 + 32;
  static constexpr int K_BYTES = kTileKeys * KROW, V_BYTES = kTileKeys * VROW;
  static constexpr int BYTES = K_BYTES + V_BYTES;  // one buffer
};

// max over the two lanes (l, l + 32) that share a query column
__device__ __forceinline__ float halves_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return vmax2(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

template <int HD> struct PrefillSmem {
  __attribute__((aligned(16))) char lds[2 * Lds<HD>::BYTES];
  int last;
};

// Eight consecutive dims of a lane's column from two accumulator quads x, y
// (dims 4 half + 0..3 and 8 + 4 half + 0..3 of a 16-dim group): after the
// exchange between the halves, half 0 holds dims 0..7 and half 1 dims 8..15.
__device__ __forceinline__ void gather8(const f32x16& acc, int e, float scale, float* o) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[e + j] * scale),
                                                    __float_as_uint(acc[e + 4 + j] * scale), false, false);
    o[j] = __uint_as_float(r[0]);
    o[4 + j] = __uint_as_float(r[1]);
  }
}

// The end of a tile: its output, or its partial and, in the last partition to
// arrive, the merge. Column tile nc of a lane holds query row row_of[nc] (-1:
// none) and head head_of[nc], accumulators acc less base, and the lane's half
// of the row sum.
template <typename ACT, typename KV, int HD, int NC>
__device__ __forceinline__ void finish_tile(const ChunkParams& p, const ChunkItem& it, int kvh, int& last,
                                            f32x16 (&acc)[NC][HD / 32], float (&base)[NC], float (&lsum)[NC],
                                            int (&row_of)[NC], int (&head_of)[NC]) {
  constexpr int DT = HD / 32;
  const int tid = threadIdx.x, half = (tid & (kWave - 1)) >> 5;
  const int G = p.q_heads / p.kv_heads;
  // acc[nc][d][e] = O[column][dim 32 d + 8 (e / 4) + 4 half + e % 4]
  float l_tot[NC];
#pragma unroll
  for (int nc = 0; nc < NC; nc++) l_tot[nc] = halves_sum(lsum[nc]);
  if (it.part0 < 0) {
#pragma unroll
    for (int nc = 0; nc < NC; nc++) {
      ACT* out = static_cast<ACT*>(p.out) +
                 (static_cast<int64_t>(it.tok_begin + max(row_of[nc], 0)) * p.q_heads + head_of[nc]) * HD + half * 8;
      const float inv = 1.f / l_tot[nc];
#pragma unroll
      for (int d = 0; d < DT; d++)
#pragma unroll
        for (int e = 0; e < 16; e += 8) {
          float f[8];
          gather8(acc[nc][d], e, inv, f);  // every lane takes part in the exchange
          if (row_of[nc] >= 0) elem<ACT>::store8(out + d * 32 + e * 2, f);
        }
    }
#ifdef LE_TIMING
    __builtin_amdgcn_s_waitcnt(0);
    LE_TIM(3, LE_TIM_NOW());
    LE_TIM(4, LE_TIM_NOW());
#endif
    return;
  }

  // ---- split tile: the partial in the chunk kernel's record layout, then
  // the last partition to arrive merges ----
  const int64_t rec_tile = static_cast<int64_t>(it.part0 - it.part) * p.q_heads;
  const __amdgpu_buffer_rsrc_t acc_rsrc = coherent_rsrc(p.parts.acc + rec_tile * HD);
  float* ml = reinterpret_cast<float*>(p.parts.ml);
#pragma unroll
  for (int nc = 0; nc < NC; nc++) {
    const bool on = row_of[nc] >= 0;
    const int64_t rec = static_cast<int64_t>(it.part0 + max(row_of[nc], 0) * it.part_stride) * p.q_heads + head_of[nc];
    const float inv = l_tot[nc] > 0.f ? 1.f / l_tot[nc] : 0.f;
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
      for (int e = 0; e < 16; e += 8) {
        float f[8];
        gather8(acc[nc][d], e, inv, f);
        if (!on) continue;
        const int64_t el = (rec - rec_tile) * HD + d * 32 + e * 2 + half * 8;
        if constexpr (chk::kHalfPartials<KV>) {
          const uint4 h = make_uint4(pack_f16x2(f[0], f[1]), pack_f16x2(f[2], f[3]), pack_f16x2(f[4], f[5]),
                                     pack_f16x2(f[6], f[7]));
          const f32x4v v = __builtin_bit_cast(f32x4v, h);
          if (p.l2_local) st_l2_16(acc_rsrc, static_cast<uint32_t>(el * 2), v);
          else st_coherent16(acc_rsrc, static_cast<uint32_t>(el * 2), v);
        } else {
#pragma unroll
          for (int q = 0; q < 2; q++) {
            const f32x4v v = {f[4 * q], f[4 * q + 1], f[4 * q + 2], f[4 * q + 3]};
            if (p.l2_local) st_l2_16(acc_rsrc, static_cast<uint32_t>((el + 4 * q) * 4), v);
            else st_coherent16(acc_rsrc, static_cast<uint32_t>((el + 4 * q) * 4), v);
          }
        }
      }
    if (on && half == 0) {
      const float m = l_tot[nc] > 0.f ? base[nc] : -FLT_MAX;
      if (p.l2_local) {
        reinterpret_cast<float2*>(ml)[rec] = make_float2(m, l_tot[nc]);
      } else {
        chk::st_dev(ml + rec * 2, m);
        chk::st_dev(ml + rec * 2 + 1, l_tot[nc]);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0);  // this thread's partial stores are performed
  __syncthreads();                // ... and every other thread's
  LE_TIM(3, LE_TIM_NOW());
  arrival_t* counter = p.parts.counters + static_cast<int64_t>(it.tok_begin) * p.kv_heads + kvh;
  if (tid == 0) {
    const arrival_t seen = __hip_atomic_fetch_add(counter, arrival_t{1}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = seen == static_cast<arrival_t>(it.part_stride - 1);
  }
  __syncthreads();
#ifdef LE_TIMING
  if (!last) LE_TIM(4, LE_TIM_NOW());
#endif
  if (!last) return;
  chk::merge_tile<ACT, HD, 4, chk::kHalfPartials<KV>, kThreads, HD == 64 && NC == 1 ? 2 : 4>(p, it, acc_rsrc, ml, rec_tile, it.part0 - it.part,
                                                               it.part_stride, G, kvh, it.n_q, it.tok_begin);
  if (tid == 0) __hip_atomic_store(counter, arrival_t{0}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#ifdef LE_TIMING
  __builtin_amdgcn_s_waitcnt(0);  // the merge's output stores are performed
  LE_TIM(4, LE_TIM_NOW());
#endif
}

// What a prefill workgroup stamps at its start (measurement builds).
__device__ __forceinline__ void stamp_item(const ChunkItem& it, uint64_t t_start) {
  LE_TIM(0, t_start);
  LE_TIM(5, LE_TIM_PLACE());
  LE_TIM(6, (static_cast<uint64_t>(it.blk_end - it.blk_begin) << 32) | static_cast<uint32_t>(it.part0 < 0 ? 0 : it.part_stride));
  LE_TIM(7, 2);
}

// The workgroup's item; n_q 0: nothing to do (padding that keeps split tiles
// on one XCD, or a partition past the first of a tile that runs whole). kWhole:
// without a list of ids there is no workspace, and split tiles run whole.
template <bool kWhole> __device__ __forceinline__ ChunkItem tile_item(const ChunkParams& p, int item) {
  ChunkItem it = p.items[item];
  if (kWhole && !p.item_ids && it.n_q > 0) {
    it.n_q = it.part == 0 ? it.n_q : 0;
    it.part0 = -1;
    it.key_live = p.token_pos[it.tok_begin] + it.n_q;
    if (it.seq >= 0) it.seq = ~p.table_offset[it.seq];
  }
  return it;
}

// The item's block ids: the plan's list, or, past its width, the sequence's
// table. Both lie in the plan's buffer: one base and a scalar offset (a choice
// between two pointers took up to 11 more VGPRs in the mixed-step kernels).
__device__ __forceinline__ const int32_t* tile_ids(const ChunkParams& p, const ChunkItem& it, int item) {
  const int64_t listed = p.item_ids - p.tables + static_cast<int64_t>(item) * p.ids_stride;
  const int64_t off = it.seq < 0 ? static_cast<int64_t>(~it.seq) + it.blk_begin : listed;
  return p.tables + __builtin_amdgcn_readfirstlane(static_cast<int>(off));
}

// One prefill workgroup: item `item`, kv head `kvh`, NC column tiles a wave.
// kWhole: p.item_ids may be null (tile_item).
template <typename ACT, typename KV, int HD, int NC, bool kWhole = false>
__device__ __forceinline__ void prefill_wg(const ChunkParams& p, PrefillSmem<HD>& sm, int item, int kvh) {
  using M = mma16<KV>;
  using V8 = typename M::v8;
  using V4 = typename M::v4;
  using S16 = typename M::scalar;
  using W = mma32<KV>;
  using L = Lds<HD>;
  static_assert(NC * kWaves * 32 == prefill_cols(NC == 2));
  constexpr int KS = HD / 16;   // k-steps of S^T
  constexpr int DT = HD / 32;   // 32-dim output tiles
  constexpr int CPR = HD / 8;   // 16-byte pieces of a K/V row
  constexpr int KPT = kTileKeys * CPR / kThreads;  // keys (one piece each) a thread moves per tile
  constexpr int KSTEP = kThreads / CPR;             // keys between them

  char* lds = sm.lds;
  int& last = sm.last;
  [[maybe_unused]] const uint64_t t_start = LE_TIM_NOW();
  const ChunkItem it = tile_item<kWhole>(p, item);
  if (it.n_q <= 0) return;
  stamp_item(it, t_start);
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int G = p.q_heads / p.kv_heads;
  const int bs_shift = __builtin_ctz(p.block_size);
  const int bs_mask = p.block_size - 1;
  const int64_t row_bytes = static_cast<int64_t>(p.kv_heads) * HD * 2;
  const int key_begin = it.blk_begin << bs_shift;
  const int32_t* ids = tile_ids(p, it, item);
  const char* kbase = static_cast<const char*>(p.k_cache) + kvh * (HD * 2);
  const char* vbase = static_cast<const char*>(p.v_cache) + kvh * (HD * 2);

  // ---- staging: this thread's piece of KPT keys per tile ----
  const int key_l = tid / CPR, piece = tid - key_l * CPR;
  struct Stage {  // one tile's loads in flight
    uint4 k[KPT], v[KPT];
    bool ok[KPT];
  };
  Stage sa, sb;
  int32_t bid[KPT];
  auto fetch_ids = [&](int rel0) {
#pragma unroll
    for (int k = 0; k < KPT; k++) bid[k] = ids[min(rel0 + key_l + k * KSTEP, it.key_live - 1) >> bs_shift];
  };
  auto issue = [&](Stage& st, int rel0) {
#pragma unroll
    for (int k = 0; k < KPT; k++) {
      const int rel = rel0 + key_l + k * KSTEP;
      const bool ok = bid[k] >= 0 && bid[k] < p.num_cache_blocks;
      st.ok[k] = ok && rel < it.key_live;
      const int slot_in = min(rel, it.key_live - 1) & bs_mask;
      const int64_t off = ((static_cast<int64_t>(ok ? bid[k] : 0) << bs_shift) + slot_in) * row_bytes + piece * 16;
      st.k[k] = ld16(kbase + off);
      st.v[k] = ld16(vbase + off);
    }
  };
  auto stash = [&](const Stage& st, int buf) {
    char* b = lds + buf * L::BYTES;
#pragma unroll
    for (int k = 0; k < KPT; k++) {
      const int key = key_l + k * KSTEP;
      *reinterpret_cast<uint4*>(b + key * L::KROW + piece * 16) = st.ok[k] ? st.k[k] : make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(b + L::K_BYTES + key * L::VROW + piece * 16) = st.ok[k] ? st.v[k] : make_uint4(0, 0, 0, 0);
    }
  };
  fetch_ids(0);

  // ---- Q^T: column c's dims ks*16 + half*8 .. +8 per k-step ----
  const int pos0 = p.token_pos[it.tok_begin];
  // (loaded raw, converted once the first tile's K/V loads are on their way)
  constexpr int QW = sizeof(ACT) / 2;  // 16-byte pieces of 8 elements
  V8 qb[NC][KS];
  uint4 qraw[NC][KS][QW];
  int lim[NC];  // position of the column's row; -1: no such row
  int row_of[NC], head_of[NC];
#pragma unroll
  for (int nc = 0; nc < NC; nc++) {
    const int c = (wave * NC + nc) * 32 + col;
    const int r = c / G;
    const bool ok = r < it.n_q;
    row_of[nc] = ok ? r : -1;
    head_of[nc] = kvh * G + (c - r * G);
    lim[nc] = ok ? pos0 + r - key_begin : -1;  // last live key, relative to key_begin
    const ACT* q = static_cast<const ACT*>(p.q) +
                   (static_cast<int64_t>(it.tok_begin + (ok ? r : 0)) * p.q_heads + head_of[nc]) * HD + half * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int h = 0; h < QW; h++) qraw[nc][ks][h] = ld16(q + ks * 16 + h * 4);
  }
  issue(sa, 0);
  fetch_ids(kTileKeys);
#pragma unroll
  for (int nc = 0; nc < NC; nc++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      float f[8];
      if constexpr (QW == 1) {
        elem<ACT>::widen(qraw[nc][ks][0], f);
      } else {
        elem<float>::widen(qraw[nc][ks][0], f);
        elem<float>::widen(qraw[nc][ks][1], f + 4);
      }
#pragma unroll
      for (int e = 0; e < 8; e++) qb[nc][ks][e] = static_cast<S16>(row_of[nc] >= 0 ? f[e] * p.scale_log2 : 0.f);
    }
  // The wave's first and last row: tiles past the last row's position hold
  // no key of the wave, tiles up to the first row's need no mask.
  const int c0 = wave * NC * 32;
  const int first_row = min(c0 / G, it.n_q - 1), last_row = min((c0 + NC * 32 - 1) / G, it.n_q - 1);
  const int wave_lim = c0 / G < it.n_q ? min(pos0 + last_row - key_begin, it.key_live - 1) : -1;
  const int free_lim = min(pos0 + first_row - key_begin, it.key_live - 1);

  f32x16 acc[NC][DT];
  // Scores leave the first product less the column's base (-base is the MFMA's
  // C operand), in log2 units; thr is what they may rise to before it moves.
  float base[NC], thr[NC], lsum[NC];
  f32x16 nbase[NC];
#pragma unroll
  for (int nc = 0; nc < NC; nc++) {
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[nc][d][e] = 0.f;
    base[nc] = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) nbase[nc][e] = 0.f;
    thr[nc] = -FLT_MAX;  // no live key yet
    lsum[nc] = 0.f;
  }
  typename W::v2 ones;
  ones[0] = static_cast<S16>(1.f);
  ones[1] = static_cast<S16>(1.f);
  // One tile of keys from LDS buffer b, its first key rel: both 32-key halves
  // together, so one half's products run beside the other's softmax (2048
  // rows after 8192, head_dim 128: 357 against 364 us half by half).
  constexpr int U = kTileKeys / 32;
  const int l16 = lane & 15;
  auto tile = [&](const char* b, int rel) {
    f32x16 s[U][NC];
    const char* kp = b + col * L::KROW + half * 16;
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        const V8 ka = *reinterpret_cast<const V8*>(kp + u * 32 * L::KROW + ks * 32);
#pragma unroll
        for (int nc = 0; nc < NC; nc++) s[u][nc] = W::mma(ka, qb[nc][ks], ks == 0 ? nbase[nc] : s[u][nc]);
      }
    // accumulator e of a lane is key 8 * (e / 4) + 4 * half + e % 4
    if (rel + 32 * U - 1 > free_lim) {
#pragma unroll
      for (int nc = 0; nc < NC; nc++) {
        const int m = min(lim[nc], it.key_live - 1) - rel - half * 4;
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int e = 0; e < 16; e++)
            if (32 * u + 8 * (e / 4) + e % 4 > m) s[u][nc][e] = -INFINITY;
      }
    }
    float mt[NC];
    bool move = false;
#pragma unroll
    for (int nc = 0; nc < NC; nc++) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        const f32x16& x = s[u][nc];
        const float m0 = chk::vmax3(x[0], x[1], x[2]), m1 = chk::vmax3(x[3], x[4], x[5]);
        const float m2 = chk::vmax3(x[6], x[7], x[8]), m3 = chk::vmax3(x[9], x[10], x[11]);
        const float m4 = chk::vmax3(x[12], x[13], x[14]);
        const float mu = vmax2(chk::vmax3(m0, m1, m2), chk::vmax3(m3, m4, x[15]));
        mt[nc] = u == 0 ? mu : vmax2(mt[nc], mu);
      }
      move |= mt[nc] > thr[nc];
    }
    if (__builtin_amdgcn_ballot_w64(move)) {
      // A column's first live keys set its base to their maximum; later keys
      // move it when they pass it by more than kRescaleSlack, and what is
      // accumulated is rescaled.
#pragma unroll
      for (int nc = 0; nc < NC; nc++) {
        const float m = halves_max(mt[nc]);
        const bool fresh = thr[nc] == -FLT_MAX;
        const bool go = m > thr[nc];
        const float shift = go ? m : 0.f;
        const float alpha = go && !fresh ? __builtin_amdgcn_exp2f(-shift) : 1.f;
        base[nc] += shift;
        thr[nc] = go ? chk::kRescaleSlack : thr[nc];
        lsum[nc] *= alpha;
#pragma unroll
        for (int d = 0; d < DT; d++) acc[nc][d] *= alpha;
#pragma unroll
        for (int e = 0; e < 16; e++) nbase[nc][e] = -base[nc];
#pragma unroll
        for (int u = 0; u < U; u++) s[u][nc] -= shift;
      }
    }
    V8 pb[U][NC][2];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int nc = 0; nc < NC; nc++) {
#pragma unroll
        for (int e = 0; e < 16; e++) pb[u][nc][e / 8][e % 8] = static_cast<S16>(__builtin_amdgcn_exp2f(s[u][nc][e]));
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
          typename W::v2 pr;
          pr[0] = pb[u][nc][e / 8][e % 8];
          pr[1] = pb[u][nc][e / 8][e % 8 + 1];
          lsum[nc] = W::dot2(pr, ones, lsum[nc]);
        }
      }
    // V^T operand of key step t: lane (dim 16 * (lane / 16 % 2) + lane % 16,
    // half) holds keys 16t + 4 half + 0..3 and 16t + 8 + 4 half + 0..3, the
    // keys of accumulators 8t .. 8t + 7
    const char* vp = b + L::K_BYTES + (4 * half + (l16 >> 2)) * L::VROW + ((lane >> 4) & 1) * 32 + (l16 & 3) * 8;
#pragma unroll
    for (int t = 0; t < 2 * U; t++)
#pragma unroll
      for (int d = 0; d < DT; d++) {
        const V4 lo = lds_read_tr16<KV>(vp + 16 * t * L::VROW + d * 64);
        const V4 hi = lds_read_tr16<KV>(vp + (16 * t + 8) * L::VROW + d * 64);
        const V8 va = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int nc = 0; nc < NC; nc++) acc[nc][d] = W::mma(va, pb[t / 2][nc][t % 2], acc[nc][d]);
      }
  };

  // kAhead tiles of loads in flight, in registers, beside the tile being
  // computed (two: 512 rows after 1024 keys, 14/2 heads x 64, 15.6 against 16.2
  // us; at head_dim 128 the second tile's registers spill: 42.5 against 39).
  constexpr int kAhead = HD == 64 ? 2 : 1;
  const int n_tiles = (it.key_live + kTileKeys - 1) / kTileKeys;
  // tile t; loads tile t + kAhead into `load` and stashes tile t + 1 from `next`
  auto step = [&](int t, Stage& load, const Stage& next) {
    const int rel = t * kTileKeys;
    if (t + kAhead < n_tiles) {
      issue(load, rel + kAhead * kTileKeys);
      fetch_ids(rel + (kAhead + 1) * kTileKeys);
    }
    if (rel <= wave_lim) tile(lds + (t & 1) * L::BYTES, rel);
    if (t + 1 < n_tiles) {
      stash(next, (t + 1) & 1);
      __syncthreads();
    }
  };
  if constexpr (kAhead == 2) {
    issue(sb, kTileKeys);  // (clamped to live keys where there is no second tile)
    fetch_ids(2 * kTileKeys);
  }
  stash(sa, 0);
  __syncthreads();
  LE_TIM(1, LE_TIM_NOW());
  if constexpr (kAhead == 2) {
    for (int t = 0; t < n_tiles; t += 2) {
      step(t, sa, sb);
      if (t + 1 < n_tiles) step(t + 1, sb, sa);
    }
  } else {
    for (int t = 0; t < n_tiles; t++) step(t, sa, sa);
  }

  LE_TIM(2, LE_TIM_NOW());
  LE_TIM_WAVE(8, LE_TIM_NOW());
  finish_tile<ACT, KV, HD, NC>(p, it, kvh, last, acc, base, lsum, row_of, head_of);
}

}  // namespace
}  // namespace pre
}  // namespace le
