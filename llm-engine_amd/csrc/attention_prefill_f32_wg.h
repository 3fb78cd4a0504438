#pragma once
// Prefill chunk rows on MFMA, fp32 caches with head_dim 64 (hot-path part 3):
// the prefill tile's workgroup.
//
// The same function and the same arithmetic as the chunk tile with an fp32
// cache (attention_chunk_wg.h: every operand in three bf16 terms, every
// product as six, fp32 softmax and row sums), in the prefill tile's shape
// (attention_prefill_wg.h: 128 packed (row, head) columns, four waves of 32,
// the 32x32x16 MFMA).
// The chunk tile (eight waves, one per query head of the group, 32 rows)
// leaves waves idle below eight heads, reads every K/V fragment for 32 rows of
// one head, and nothing overlaps its stores to LDS. Chunk tile against this
// one (us per call): 4096 rows after 0-1536 keys, 32/4 heads x 64, 286 against
// 225 (0.92 PFLOP/s of bf16 products); 2048 rows after 8192, 982 against 855;
// 4 x 200 rows after 300, 16/16 heads, 78 against 28; 40 rows after 8000, 140
// against 59; 3 x 333 rows after 0-700 with 5 decode rows and the K/V store,
// 14/2 heads, 45.6 against 38.8. Error against 64 bits in the last 3.8e-7
// (chunk tile 4.1e-7).
//
//   * 64-key tiles, single buffered: the three planes of K and V take 58 KB, so
//     two workgroups share a CU and one's matrix work runs beside the other's
//     split and softmax. The next tile's loads are in flight in registers
//     during a tile's products.
//   * a wave reads 48 KB of fragments from LDS and issues 96 MFMAs (3072
//     cycles) a tile: the matrix cores bound it while there is a workgroup for
//     every slot, the tile's serial chain below that.
#include "attention_prefill_wg.h"

namespace le {
namespace pre {
namespace {

template <int HD> struct LdsF32 {
  static constexpr int KROW = HD * 2 + 16, VROW = HD * 2 + 32;  // of one plane, padded as in Lds
  static constexpr int KPLANE = kTileKeys * KROW, VPLANE = kTileKeys * VROW;
  static constexpr int BYTES = 3 * (KPLANE + VPLANE);  // K planes hi, mid, lo, then V's
};

template <int HD> struct PrefillF32Smem {
  __attribute__((aligned(16))) char lds[LdsF32<HD>::BYTES];
  int last;
};

// One prefill workgroup of an fp32 cache: item `item`, kv head `kvh`.
template <typename ACT, int HD, bool kWhole = false>
__device__ __forceinline__ void prefill_f32_wg(const ChunkParams& p, PrefillF32Smem<HD>& sm, int item, int kvh) {
  using M = mma16<bf16_t>;
  using V8 = typename M::v8;
  using V4 = typename M::v4;
  using W = mma32<bf16_t>;
  using L = LdsF32<HD>;
  constexpr int KS = HD / 16;   // k-steps of S^T
  constexpr int DT = HD / 32;   // 32-dim output tiles
  constexpr int CPR = HD / 4;   // 16-byte pieces of a K/V row
  constexpr int KPT = kTileKeys * CPR / kThreads;  // keys (one piece each) a thread moves per tile
  constexpr int KSTEP = kThreads / CPR;             // keys between them
  constexpr int U = kTileKeys / 32;

  char* lds = sm.lds;
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
  const int64_t row_bytes = static_cast<int64_t>(p.kv_heads) * HD * 4;
  const int key_begin = it.blk_begin << bs_shift;
  const int32_t* ids = tile_ids(p, it, item);
  const char* kbase = static_cast<const char*>(p.k_cache) + kvh * (HD * 4);
  const char* vbase = static_cast<const char*>(p.v_cache) + kvh * (HD * 4);

  // ---- staging: this thread's piece of KPT keys per tile ----
  const int key_l = tid / CPR, piece = tid - key_l * CPR;
  uint4 sk[KPT], sv[KPT];
  bool ok[KPT];
  int32_t bid[KPT];
  auto fetch_ids = [&](int rel0) {
#pragma unroll
    for (int k = 0; k < KPT; k++) bid[k] = ids[min(rel0 + key_l + k * KSTEP, it.key_live - 1) >> bs_shift];
  };
  auto issue = [&](int rel0) {
#pragma unroll
    for (int k = 0; k < KPT; k++) {
      const int rel = rel0 + key_l + k * KSTEP;
      const bool valid = bid[k] >= 0 && bid[k] < p.num_cache_blocks;
      ok[k] = valid && rel < it.key_live;
      const int slot_in = min(rel, it.key_live - 1) & bs_mask;
      const int64_t off = ((static_cast<int64_t>(valid ? bid[k] : 0) << bs_shift) + slot_in) * row_bytes + piece * 16;
      sk[k] = ld16(kbase + off);
      sv[k] = ld16(vbase + off);
    }
  };
  // four fp32 dims become 8 bytes in each of the three planes; a dead key's are zeros
  auto put = [&](char* dst, int plane, const uint4& raw, bool live) {
    const uint4 u = live ? raw : make_uint4(0, 0, 0, 0);
    const float f[4] = {__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w)};
    V4 h, m, l;
#pragma unroll
    for (int e = 0; e < 4; e++) chk::put3(h, m, l, e, f[e]);
    *reinterpret_cast<V4*>(dst) = h;
    *reinterpret_cast<V4*>(dst + plane) = m;
    *reinterpret_cast<V4*>(dst + 2 * plane) = l;
  };
  auto stash = [&]() {
#pragma unroll
    for (int k = 0; k < KPT; k++) {
      const int key = key_l + k * KSTEP;
      put(lds + key * L::KROW + piece * 8, L::KPLANE, sk[k], ok[k]);
      put(lds + 3 * L::KPLANE + key * L::VROW + piece * 8, L::VPLANE, sv[k], ok[k]);
    }
  };
  fetch_ids(0);

  // ---- Q^T: column c's dims ks*16 + half*8 .. +8 per k-step, three terms ----
  const int pos0 = p.token_pos[it.tok_begin];
  constexpr int QW = sizeof(ACT) / 2;  // 16-byte pieces of 8 elements
  V8 qh[KS], qm[KS], ql[KS];
  uint4 qraw[KS][QW];
  const int c = wave * 32 + col;
  const int r = c / G;
  int row_of[1] = {r < it.n_q ? r : -1};
  int head_of[1] = {kvh * G + (c - r * G)};
  const int lim = row_of[0] >= 0 ? pos0 + r - key_begin : -1;  // last live key, relative to key_begin
  {
    const ACT* q = static_cast<const ACT*>(p.q) +
                   (static_cast<int64_t>(it.tok_begin + max(row_of[0], 0)) * p.q_heads + head_of[0]) * HD + half * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int h = 0; h < QW; h++) qraw[ks][h] = ld16(q + ks * 16 + h * 4);
  }
  issue(0);
  fetch_ids(kTileKeys);
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    float f[8];
    if constexpr (QW == 1) {
      elem<ACT>::widen(qraw[ks][0], f);
    } else {
      elem<float>::widen(qraw[ks][0], f);
      elem<float>::widen(qraw[ks][1], f + 4);
    }
#pragma unroll
    for (int e = 0; e < 8; e++) chk::put3(qh[ks], qm[ks], ql[ks], e, row_of[0] >= 0 ? f[e] * p.scale_log2 : 0.f);
  }
  // Tiles past the wave's last row's position hold no key of the wave, tiles
  // up to its first row's need no mask.
  const int c0 = wave * 32;
  const int first_row = min(c0 / G, it.n_q - 1), last_row = min((c0 + 31) / G, it.n_q - 1);
  const int wave_lim = c0 / G < it.n_q ? min(pos0 + last_row - key_begin, it.key_live - 1) : -1;
  const int free_lim = min(pos0 + first_row - key_begin, it.key_live - 1);

  // as in prefill_wg: scores leave the first product less the column's base
  f32x16 acc[1][DT], nbase;
  float base[1] = {0.f}, lsum[1] = {0.f}, thr = -FLT_MAX;
#pragma unroll
  for (int e = 0; e < 16; e++) {
    nbase[e] = 0.f;
#pragma unroll
    for (int d = 0; d < DT; d++) acc[0][d][e] = 0.f;
  }
  const int l16 = lane & 15;
  auto tile = [&](int rel) {
    f32x16 s[U];
    const char* kp = lds + col * L::KROW + half * 16;
#pragma unroll
    for (int u = 0; u < U; u++) s[u] = nbase;
    // per 16 dims: the key halves' three terms, their six products each,
    // smallest terms first
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      V8 kh[U], km[U], kl[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const char* k = kp + u * 32 * L::KROW + ks * 32;
        kh[u] = *reinterpret_cast<const V8*>(k);
        km[u] = *reinterpret_cast<const V8*>(k + L::KPLANE);
        kl[u] = *reinterpret_cast<const V8*>(k + 2 * L::KPLANE);
      }
#pragma unroll
      for (int u = 0; u < U; u++) s[u] = W::mma(kl[u], qh[ks], s[u]);
#pragma unroll
      for (int u = 0; u < U; u++) s[u] = W::mma(km[u], qm[ks], s[u]);
#pragma unroll
      for (int u = 0; u < U; u++) s[u] = W::mma(kh[u], ql[ks], s[u]);
#pragma unroll
      for (int u = 0; u < U; u++) s[u] = W::mma(km[u], qh[ks], s[u]);
#pragma unroll
      for (int u = 0; u < U; u++) s[u] = W::mma(kh[u], qm[ks], s[u]);
#pragma unroll
      for (int u = 0; u < U; u++) s[u] = W::mma(kh[u], qh[ks], s[u]);
    }
    // accumulator e of a lane is key 8 * (e / 4) + 4 * half + e % 4
    if (rel + kTileKeys - 1 > free_lim) {
      const int m = min(lim, it.key_live - 1) - rel - half * 4;
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int e = 0; e < 16; e++)
          if (32 * u + 8 * (e / 4) + e % 4 > m) s[u][e] = -INFINITY;
    }
    float mt = -INFINITY;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const f32x16& x = s[u];
      const float m0 = chk::vmax3(x[0], x[1], x[2]), m1 = chk::vmax3(x[3], x[4], x[5]);
      const float m2 = chk::vmax3(x[6], x[7], x[8]), m3 = chk::vmax3(x[9], x[10], x[11]);
      const float m4 = chk::vmax3(x[12], x[13], x[14]);
      mt = vmax2(mt, vmax2(chk::vmax3(m0, m1, m2), chk::vmax3(m3, m4, x[15])));
    }
    if (__builtin_amdgcn_ballot_w64(mt > thr)) {
      const float m = halves_max(mt);
      const bool fresh = thr == -FLT_MAX;
      const bool go = m > thr;
      const float shift = go ? m : 0.f;
      const float alpha = go && !fresh ? __builtin_amdgcn_exp2f(-shift) : 1.f;
      base[0] += shift;
      thr = go ? chk::kRescaleSlack : thr;
      lsum[0] *= alpha;
#pragma unroll
      for (int d = 0; d < DT; d++) acc[0][d] *= alpha;
#pragma unroll
      for (int e = 0; e < 16; e++) nbase[e] = -base[0];
#pragma unroll
      for (int u = 0; u < U; u++) s[u] -= shift;
    }
    const char* vp = lds + 3 * L::KPLANE + (4 * half + (l16 >> 2)) * L::VROW + ((lane >> 4) & 1) * 32 + (l16 & 3) * 8;
#pragma unroll
    for (int t = 0; t < 2 * U; t++) {  // 16 keys: accumulators 8 (t % 2) .. + 8 of half t / 2
      V8 ph, pm, pl;
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        x[e] = __builtin_amdgcn_exp2f(s[t / 2][8 * (t % 2) + e]);
        chk::put3(ph, pm, pl, e, x[e]);
      }
      lsum[0] += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
      V8 v[DT][3];
#pragma unroll
      for (int d = 0; d < DT; d++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const V4 lo = lds_read_tr16<bf16_t>(vp + i * L::VPLANE + 16 * t * L::VROW + d * 64);
          const V4 hi = lds_read_tr16<bf16_t>(vp + i * L::VPLANE + (16 * t + 8) * L::VROW + d * 64);
          v[d][i] = V8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
#pragma unroll
      for (int d = 0; d < DT; d++) acc[0][d] = W::mma(v[d][2], ph, acc[0][d]);
#pragma unroll
      for (int d = 0; d < DT; d++) acc[0][d] = W::mma(v[d][1], pm, acc[0][d]);
#pragma unroll
      for (int d = 0; d < DT; d++) acc[0][d] = W::mma(v[d][0], pl, acc[0][d]);
#pragma unroll
      for (int d = 0; d < DT; d++) acc[0][d] = W::mma(v[d][1], ph, acc[0][d]);
#pragma unroll
      for (int d = 0; d < DT; d++) acc[0][d] = W::mma(v[d][0], pm, acc[0][d]);
#pragma unroll
      for (int d = 0; d < DT; d++) acc[0][d] = W::mma(v[d][0], ph, acc[0][d]);
    }
  };

  const int n_tiles = (it.key_live + kTileKeys - 1) / kTileKeys;
  for (int t = 0; t < n_tiles; t++) {
    const int rel = t * kTileKeys;
    stash();
    __syncthreads();
    if (t == 0) LE_TIM(1, LE_TIM_NOW());
    if (t + 1 < n_tiles) {
      issue(rel + kTileKeys);
      fetch_ids(rel + 2 * kTileKeys);
    }
    if (rel <= wave_lim) tile(rel);
    if (t + 1 < n_tiles) __syncthreads();  // the tile is no longer read
  }
  LE_TIM(2, LE_TIM_NOW());
  LE_TIM_WAVE(8, LE_TIM_NOW());
  finish_tile<ACT, float, HD, 1>(p, it, kvh, sm.last, acc, base, lsum, row_of, head_of);
}

}  // namespace
}  // namespace pre
}  // namespace le
