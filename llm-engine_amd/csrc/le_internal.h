// Internal launch functions behind the C ABI in include/llm_engine_amd.h.
// Argument validation happens in abi.cpp; these assume valid shapes.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace le {

// Split-K partial result of one (row, q head, context partition): the
// unnormalised accumulator, and the running max (log2 domain) and sum.
struct PartialLayout {
  float* acc;         // [n_parts][q_heads][head_dim]
  float2* ml;         // [n_parts][q_heads]  (m, l)
  unsigned long long* counters;  // [n_rows][kv_heads] arrivals; zero between launches
};

// Decode work item: query row `token` (position `pos`, block table starting
// at tables + table_off) over blocks [blk_begin, blk_end) of its table. The
// row's position and table offset travel in the item so a workgroup reaches
// its first K/V load after one dependent read. part < 0: the row has a single
// partition and the kernel writes the normalised output itself. Otherwise the
// item writes partial `part`, and the last of the row's n_parts items to
// arrive (per kv head) merges partials [part_begin, part_begin + n_parts).
struct DecodeItem {
  int32_t token, pos, table_off, blk_begin, blk_end, part, part_begin, n_parts;
};

// Chunk work item: query rows [tok_begin, tok_begin + n_q) (consecutive
// positions of one sequence, at most 32, or prefill_rows() of a prefill tile)
// over key blocks [blk_begin, blk_end)
// of its table, partition `part` of the tile's part_stride partitions. Row
// tok_begin + i writes partial part0 + i * part_stride, or, when part0 < 0,
// its normalised output directly; the last partition of the tile to arrive
// (per kv head) merges partials [part0 - part + i * part_stride, ... +
// part_stride) of each row.
// seq is the sequence's index, or, of a prefill tile with more block ids than
// are listed with the item, ~ where its table starts.
struct ChunkItem {
  int32_t tok_begin, n_q, blk_begin, blk_end, part0, part_stride, seq, part;
  // keys of [blk_begin * block_size, ...) that hold a live position (at most
  // the tile's last position + 1): rows past it are never read
  int32_t key_live;
};

// Element types are passed as le_dtype codes: 0 fp32, 1 bf16, 2 fp16.
constexpr int kDtF32 = 0, kDtBF16 = 1, kDtF16 = 2;

hipError_t kv_cache_write(const void* k, const void* v, int src_dtype, const int32_t* slots,
                          void* kc, void* vc, int cache_dtype, int n_tokens, int kv_dim,
                          int64_t num_slots, hipStream_t stream);
hipError_t rope_kv_cache_write(const void* qkv, int act_dtype, int64_t row_stride, const float* bias,
                               const int32_t* positions, const int32_t* slots, const float* cos_t,
                               const float* sin_t, int max_pos, int n_tokens, int q_heads,
                               int kv_heads, int head_dim, void* q_out, void* kc, void* vc,
                               int cache_dtype, int64_t num_slots, hipStream_t stream,
                               const void* rms_x = nullptr, int rms_hidden = 0, float rms_eps = 0.f);

struct DecodeParams {
  const void* q;
  const void* k_cache;
  const void* v_cache;
  const int32_t* tables;
  const int32_t* table_offset;
  const int32_t* token_seq;
  const int32_t* token_pos;
  void* out;
  PartialLayout parts;
  // With a plan and a pure decode step: the step's new K/V rows ([n_tokens]
  // [kv_heads * head_dim], element type new_dtype). The last partition
  // of each row stores its row (for its kv head) at slots[token] before any
  // K/V load of the launch reads it. Null: the rows are already in the cache.
  const void* k_new;
  const void* v_new;
  const int32_t* slots;
  int new_dtype;
  int64_t num_slots;
  // Rows straight from the stacked QKV projection (rope_max_pos > 0): q and
  // the new K/V rows are read at rope_row_stride elements per token (q, k_new
  // and v_new point at row 0's q, k and v parts, all in the activation type);
  // the bias (fp32 [q | k | v], may be null) is added and rounded to the
  // activation type, then q and k rotate by the row's position (tables
  // [rope_max_pos][head_dim / 2]) exactly as rope_kv_cache_write computes
  // them. A row whose position is outside the tables attends with q = 0 and
  // stores nothing (as rope_kv_cache_write writes zeros and skips the store).
  int64_t rope_row_stride;
  const float* rope_bias;
  const float* rope_cos;
  const float* rope_sin;
  int rope_max_pos;
  // With rope rows: the pre-attention RMSNorm folded into the QKV projection.
  // rms_x (act dtype, [tokens][rms_hidden]) is the residual stream the rows
  // were projected from; each row is scaled by 1/sqrt(mean(x^2) + rms_eps)
  // before its bias. Null: the rows are already normalised.
  const void* rms_x;
  int rms_hidden;
  float rms_eps;
  const DecodeItem* items;  // null: one item per (token, split) with `nsplit` splits
  // With items: block ids of item i at item_ids[i * ids_stride + j]. Null: a
  // mixed step without a workspace; the first item of each row takes the whole
  // row, the others leave.
  const int32_t* item_ids;
  int ids_stride;
  int n_rows;               // items, or tokens when items is null
  int nsplit;
  int min_part;             // items null: least keys of a partition
  int q_heads, kv_heads, head_dim, block_size;
  float scale_log2;         // softmax scale * log2(e)
  int64_t num_cache_blocks;
  // With items: every partition of a split row runs on one XCD (the plan's
  // placement, and the dealing confirmed on this device by
  // xcd_placement_holds), so partials go through that XCD's L2 with plain
  // stores.
  int l2_local;
  // Two even rounds of one workgroup per CU or more (a plan of at least 512
  // workgroups with no empty fixed-layout slots): the decode kernel
  // instantiation with no register bound. Otherwise two workgroups per CU.
  int wide;
};

// True when this device deals a launch's workgroups to its XCDs round robin
// (workgroups whose linear ids are equal modulo 8 share an XCD): checked
// once per device with a probe launch, then cached. False while the stream
// is being captured and the device is not checked yet, or on any error.
bool xcd_placement_holds(hipStream_t stream);

hipError_t attention_decode(const DecodeParams& p, int act_dtype, int kv_dtype, hipStream_t stream);

struct ChunkParams {
  const void* q;
  const void* k_cache;
  const void* v_cache;
  const int32_t* tables;
  const int32_t* table_offset;
  const int32_t* token_pos;
  void* out;
  PartialLayout parts;
  const ChunkItem* items;
  // block ids of item i at item_ids[i * ids_stride + j] (its seq < 0: in the
  // tables). Null (prefill tiles): no workspace; the first item of each tile
  // takes the whole tile, the others leave.
  const int32_t* item_ids;
  int ids_stride;
  int n_items;
  int q_heads, kv_heads, head_dim, block_size;
  float scale_log2;
  int64_t num_cache_blocks;
  int l2_local;  // split tiles' partitions share an XCD: partials through its L2 (as DecodeParams)
};

// cfg.chunk_partition_tokens of a plan whose split rows and tiles may run
// whole, for a caller without a workspace (as an input, the default).
constexpr int kMayRunWhole = -1;

hipError_t attention_chunk(const ChunkParams& p, int act_dtype, int kv_dtype, hipStream_t stream);

// Chunk rows as prefill tiles (attention_prefill.hip; 16-bit caches and fp32 ones of head_dim 64): an item
// holds prefill_rows() consecutive rows. A plan whose chunk items are such tiles leaves
// cfg.chunk_q_tile at kPrefillTiles or kWidePrefillTiles (an explicit row tile
// is 16 or 32; as an input, both mean the default).
constexpr int kPrefillTiles = 0, kWidePrefillTiles = -1;
constexpr int prefill_cols(bool wide) { return wide ? 256 : 128; }  // query columns of a tile
constexpr int prefill_rows(bool wide, int group) { return prefill_cols(wide) / group; }
hipError_t attention_prefill(const ChunkParams& p, bool wide, int act_dtype, int kv_dtype, hipStream_t stream);

// A mixed step's chunk rows and decode rows (plan items) in one
// launch: chunk workgroups first, then decode workgroups.
hipError_t attention_ragged_prefill(const DecodeParams& d, const ChunkParams& c, bool wide, int act_dtype,
                                    int kv_dtype, hipStream_t stream);
hipError_t attention_ragged(const DecodeParams& d, const ChunkParams& c, int act_dtype, int kv_dtype,
                            hipStream_t stream);

// Split count for the reference-shaped entry point, where the host does not
// know the context lengths: enough workgroups to cover the chip several times.
int decode_nsplit(int n_tokens, int kv_heads);

// The least keys of a partition there (resolve() in attention_decode_wg.h); rows =
// tokens x kv heads. A partition has to stream for longer than its finish takes
// (partial, arrival, merge), but a chip with idle CUs gains from short ones, and
// one that the rows fill by themselves from whole rows. Measured (us a call):
// * below 128 rows 256 keys against 512: 7 rows of 1-1674, bf16, 32/8 heads x 128,
//   10.9 and 14.2; 48 of 32-2048, fp32, 14/2 x 64, 16.5 and 22.5 (128 keys 24.2
//   against 22.5 with two layers).
// * from 128 rows on 512 against 256: 24 of 100-3000, fp16, 32/8 x 128, 46.0 and
//   53.1; 116 of 348, fp32, 14/2 x 64, 26.7 and 31.0.
// * from 512 rows on 1024 against 512: 256 of 64-2048, fp16, 14/2 x 64, 41.2 and
//   44.7; 63 of 200-2000, bf16, 16/16 x 64, 63.2 and 69.1.
// * half of that for fp32 keys of head_dim 128 (1 KB each): 256 against 512 for 19
//   rows of 316-2531, 8/8 heads, 146 and 176; below 128 rows 256 stay (8 rows of
//   3736, 28/4 heads, 80.3 against 88.7 with 128).
constexpr int unplanned_part(int64_t rows, int head_dim, int kv_dtype) {
  const int keys = rows < 128 ? 256 : rows < 512 ? 512 : 1024;
  return rows >= 128 && kv_dtype == 0 /* LE_F32 */ && head_dim == 128 ? keys / 2 : keys;
}

}  // namespace le
