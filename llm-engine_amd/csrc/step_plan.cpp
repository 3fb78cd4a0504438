// Ragged step packing (hot-path part 1): le_plan_step / le_plan_upload.
//
// Reference: CudaModel::flatten and upload_step_indices,
// src/model/cuda/cuda_model.cu:434-491, and the CPU twin cpu_model.cpp:107-118.
// The reference builds five int arrays and sends them with six synchronous
// pageable cudaMemcpy calls per step, deduplicating sequences with an O(N*S)
// scan. Here the same arrays (identical values: token ids, positions, int32
// slots, token->sequence index in first-seen order, concatenated tables and
// their offsets) are written into one caller-owned buffer together with
// cu_seqlens_q / seq_lens_k and the attention work lists, then sent with one
// hipMemcpyAsync that every layer of the step shares.
//
// Work lists. A row whose slice has length 1 is a decode row: its context
// 0..pos is cut into partitions of ~partition_tokens (whole blocks, equal
// shares) and each partition becomes one DecodeItem. The rows of a longer
// slice (a prefill chunk) are cut into tiles of chunk_q_tile consecutive
// positions; each tile's keys 0..last position are cut into partitions of
// ~chunk_partition_tokens, one ChunkItem each, run on MFMA tiles (16-bit
// operands with a bf16/fp16 cache, fp32 operands with an fp32 cache). With
// neither size given, and a 16-bit cache or an fp32 one of head_dim 64, the
// tiles are prefill tiles instead (cut_prefill below). Split rows of either
// kind are merged inside their launch by the last partition to finish.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <unordered_map>
#include <vector>

#include "le_internal.h"
#include "llm_engine_amd.h"

namespace {

constexpr int kDefaultPartition = 640;       // decode rows: smallest automatic partition
constexpr int kSmallStepPartF32 = 256;       // fp32 cache: the smallest in a step with a CU for every workgroup
constexpr int kMaxAutoPartition = 4096;      // decode rows: largest automatic partition
constexpr int kMixedStepPartition = 2048;    // decode rows beside chunk rows: smallest automatic partition
constexpr int kPartitionQuantum = 128;       // 4 waves x 32-key fp32 tiles
constexpr int64_t kTargetItems = 512;        // workgroups per step the sizing aims for (two per CU)
constexpr int kMaxMergeEntries = 1024;       // partitions x group of one decode row (bounds the merge's loads)
constexpr int kDefaultChunkTile = 32;        // query rows per chunk item (two MFMA row tiles)
// Keys per chunk item: one and a half LDS stages. In the one-launch mixed
// step, fewer chunk workgroups leave CUs to the decode rows from the start,
// and fewer partials shorten the tiles' merges (config 3: 256 keys 24.1 us,
// 320 25.1, 384 22.7, 448 23.4, 512 25.0, 768 31.1).
constexpr int kDefaultChunkPartition = 384;
constexpr int kMaxChunkParts = 16;           // partitions of a chunk tile the in-kernel merge stages
constexpr int kMaxChunkItemBlocks = 1024;
constexpr int64_t kPrefillSlots = 512;       // prefill workgroups in flight: two per CU
constexpr int64_t kSmallPrefill = 128;       // prefill workgroups of a small step
constexpr int kSmallPrefillPart = 256;       // its smallest partition
constexpr int kPrefillSplitKeys = 576;       // shortest prefill tile worth splitting
constexpr int kMixedPrefillPartition = 1024; // decode rows beside prefill tiles: smallest automatic partition
constexpr int64_t kSmallPrefillScratch = 8 << 20;  // bytes of partials a small step may use
constexpr int kF32PrefillPart = 128;         // smallest partition of an fp32 prefill tile: two key tiles
constexpr int64_t kF32PrefillScratch = 16 << 20;    // the same with an fp32 cache
constexpr int64_t kFinerPrefillScratch = 24 << 20;  // bytes of the tiles' partials up to which decode rows split finer
constexpr int64_t kArrivalCounters = 65536;  // (row, kv head) arrival counters of a workspace
constexpr int kTileListIds = 128;            // block ids of a prefill tile that are listed beside the decode items
constexpr int kXcds = 8;                     // MI355X: XCDs, each with its own L2
constexpr int kItemOverheadBlocks = 8;       // a decode item's fixed cost, in streamed blocks    // block ids of one chunk item the kernel stages

int64_t align256(int64_t x) { return (x + 255) & ~static_cast<int64_t>(255); }

int round_to_blocks(int tokens, int bs) {
  const int b = (tokens + bs - 1) / bs;
  return b < 1 ? 1 : b;
}

// The dispatcher deals a launch's workgroups to the XCDs round robin, so
// workgroups whose linear ids are equal modulo 8 share an XCD, and each XCD
// has its own L2. The partitions of a split chunk tile (always) and of a
// split decode row (LE_PLAN_XCD_LOCAL) are kept on one XCD: the groups (one
// tile's or row's partitions) are dealt longest-first into kXcds bins, each
// to the bin with the least work so far, and item k of bin b goes to index
// k * kXcds + b. Bins are padded to one length with empty items, so the item
// count is a multiple of kXcds and the kv head's offset in the grid (a
// multiple of the item count) keeps every group on its bin's XCD.
template <typename Item, typename Same, typename Blocks>
std::vector<Item> place_on_xcds(const std::vector<Item>& items, Same same_group, Blocks blocks, const Item& pad) {
  struct Group { size_t first, n; int64_t longest, work; };
  std::vector<Group> groups;
  groups.reserve(items.size());
  for (size_t i = 0; i < items.size();) {
    size_t j = i;
    Group g{i, 0, 0, 0};
    while (j < items.size() && same_group(items[j], items[i])) {
      const int64_t nb = blocks(items[j]);
      g.longest = std::max(g.longest, nb);
      g.work += nb + kItemOverheadBlocks;
      j++;
    }
    g.n = j - i;
    groups.push_back(g);
    i = j;
  }
  // longest first; among equally long, the groups with more partitions (the
  // longer merge) first: low ids are dispatched first
  std::stable_sort(groups.begin(), groups.end(), [](const Group& a, const Group& b) {
    return a.longest != b.longest ? a.longest > b.longest : a.n > b.n;
  });
  std::vector<std::vector<Item>> bins(kXcds);
  for (auto& b : bins) b.reserve(items.size() / kXcds + 8);
  int64_t load[kXcds] = {};
  for (const Group& g : groups) {
    int b = 0;
    for (int k = 1; k < kXcds; k++)
      if (load[k] < load[b]) b = k;
    load[b] += g.work;
    for (size_t k = 0; k < g.n; k++) bins[b].push_back(items[g.first + k]);
  }
  size_t len = 0;
  for (const auto& b : bins) len = std::max(len, b.size());
  std::vector<Item> out(len * kXcds, pad);
  for (int b = 0; b < kXcds; b++)
    for (size_t k = 0; k < bins[b].size(); k++) out[k * kXcds + b] = bins[b][k];
  return out;
}

std::vector<le::DecodeItem> place_decode_items(const std::vector<le::DecodeItem>& dec) {
  le::DecodeItem pad{};
  pad.token = -1;
  pad.part = -1;
  pad.n_parts = 0;  // resolved as no work
  return place_on_xcds(
      dec, [](const le::DecodeItem& a, const le::DecodeItem& b) { return a.token == b.token && a.part_begin == b.part_begin; },
      [](const le::DecodeItem& d) { return static_cast<int64_t>(d.blk_end - d.blk_begin); }, pad);
}

std::vector<le::ChunkItem> place_chunk_items(const std::vector<le::ChunkItem>& chk) {
  le::ChunkItem pad{};
  pad.n_q = 0;  // no rows: the workgroup returns at once
  pad.part0 = -1;
  return place_on_xcds(
      chk, [](const le::ChunkItem& a, const le::ChunkItem& b) { return a.tok_begin == b.tok_begin; },
      [](const le::ChunkItem& c) { return static_cast<int64_t>(c.blk_end - c.blk_begin); }, pad);
}

// ---- prefill tiles (attention_prefill_wg.h) ----
// How a step's chunk rows are cut for the prefill kernel: tiles of `rows`
// query rows, partitions of about `part` keys (0: no tile is split).
struct PrefillCut {
  bool on = false, wide = false;
  int rows = 0;
  int64_t part = 0;
  int64_t split_keys = kPrefillSplitKeys;
  int64_t bytes = 0;  // at most this much for the tiles' partials
  // Partitions (whole blocks) of a tile over nb key blocks of bs; with `part` at
  // least kDefaultChunkPartition, no more than a 32-row tile with that end takes.
  int parts(int64_t nb, int bs) const {
    if (part == 0 || nb * bs <= split_keys) return 1;
    const int64_t pb = std::max((part + bs - 1) / bs, (nb + kMaxChunkParts - 1) / kMaxChunkParts);
    return static_cast<int>((nb + pb - 1) / pb);
  }
};

template <typename F>  // f(key blocks of the tile)
void for_prefill_tiles(const le_step_slice* s, int n, int rows, int bs, F&& f) {
  for (int i = 0; i < n; i++)
    if (s[i].len > 1)
      for (int q0 = 0; q0 < s[i].len; q0 += rows) f((s[i].start + std::min(q0 + rows, s[i].len) + bs - 1) / bs);
}

// Steps with no explicit tile or partition size, with a 16-bit cache or an fp32
// cache of head_dim 64: the prefill kernel is the faster one over all of them
// (32-row tiles against prefill tiles, us: 64 rows after 8000 keys, 32/4 heads x 64, 64 and 29; 4096
// rows after 0-1536, 131 and 63; 2048 rows after 8192, 32/8 x 128, 845 and 357;
// 512 rows after 1024, 14/2 x 64, 18.5 and 15.4; even at 1-64 rows after
// nothing, 10 and 10).
// * wide tiles (256 columns, head_dim 64): the K/V fragments a wave reads
//   from LDS serve twice the columns, but a tile takes longer and there are
//   half as many. Better from about 1000 keys per slot on (8 x 512 rows after
//   4096, 32/4 heads: 163 against 182 us; 4 x 512 after 1024: 42 against 38).
// * partitions: none when the tiles alone give three workgroups for every
//   four slots; otherwise the smallest partition that fits every workgroup
//   into the slots (the padding of the XCD placement counted), at least 384
//   keys: a split costs its partials' round trip (8 x 512 rows after 2048
//   keys: 97 us whole, 138 in 1024-key partitions). Small steps, with at most
//   kSmallPrefill workgroups, go down to 256 keys (16 rows after 1000 keys:
//   13.6 against 15.5 us; 2 x 512 rows beside 32 decode rows lose: 44 against
//   38 for two layers). Partitions below 384 keys only while their partials and
//   the decode rows' stay within kFinerPrefillScratch, so that a step which the
//   32-row tiles run in the static scratch still does.
// * an fp32 cache's tile takes six times the matrix work of a 16-bit one, so
//   splitting pays earlier: partitions of 128 keys on, the smallest that fits
//   the slots, for tiles of more than one and a half of them (16 rows after
//   1000 keys, 14/2 heads x 64: 18.2 us in 128-key partitions, 20.9 in 192, 22.2
//   in 256, 36.5 on the 32-row tiles; 300 rows after nothing 16.2, 21.3, 21.3
//   and 31.1; 512 after 1024 35.2, 35.3, 38.0 and 42.8; 4 x 200 after 300, 16/16
//   heads, 28.5, 28.5, 24.4 and 78).
// Steps with more rows than arrival counters keep the 32-row tiles: a step
// that splits nothing there runs without a workspace, and one that does is
// refused, whichever tiles would run it. (Prefill tiles that stay whole use no
// counter, so such steps could run on them: 4096 rows and 16 kv heads are the
// limit, and one decode row more takes the slower tiles.)
PrefillCut cut_prefill(const le_plan_config& cfg, const le_step_slice* s, int n, int64_t n_tok) {
  PrefillCut c;
  const int group = cfg.q_heads / cfg.kv_heads, bs = cfg.block_size;
  const bool f32 = cfg.kv_dtype == LE_F32;
  if (cfg.chunk_q_tile > 0 || cfg.chunk_partition_tokens > 0 || (f32 && cfg.head_dim != 64) ||
      (cfg.flags & LE_PLAN_TWO_LAUNCHES) || (cfg.head_dim != 64 && cfg.head_dim != 128) || group < 1 || group > 8 ||
      n_tok * cfg.kv_heads > kArrivalCounters)
    return c;
  int64_t tiles = 0, longest = 0;
  auto total_keys = [&] {  // times kv heads
    int64_t nb = 0;
    tiles = 0;
    for_prefill_tiles(s, n, c.rows, bs, [&](int64_t b) {
      nb += b;
      longest = std::max(longest, b);
      tiles++;
    });
    return nb * bs * cfg.kv_heads;
  };
  c.rows = le::prefill_rows(true, group);
  int64_t keys = total_keys();
  if (tiles == 0) return c;
  c.on = true;
  c.wide = cfg.head_dim == 64 && !f32 && keys >= 1000 * kPrefillSlots;
  c.rows = le::prefill_rows(c.wide, group);
  if (!c.wide) keys = total_keys();
  if (tiles * cfg.kv_heads * 4 >= kPrefillSlots * 3) return c;
  const int64_t padded = cfg.kv_heads % kXcds == 0 ? tiles : (tiles + kXcds - 1) / kXcds * kXcds;
  auto workgroups = [&] {  // with partitions of c.part keys; sets c.bytes
    int64_t items = 0, rows = 0;
    for_prefill_tiles(s, n, c.rows, bs, [&](int64_t b) {
      const int J = c.parts(b, bs);
      items += J;
      if (J > 1) rows += c.rows * J;
    });
    c.bytes = rows * cfg.q_heads * (cfg.head_dim * 4 + 8);
    return (items * padded + tiles - 1) / tiles * cfg.kv_heads;
  };
  int64_t decode_bytes = 0;  // the decode rows' partials
  for (int i = 0; i < n; i++)
    if (s[i].len == 1) {
      const int64_t pt = cfg.partition_tokens > 0 ? cfg.partition_tokens : kMixedPrefillPartition;
      if (s[i].start >= pt) decode_bytes += (s[i].start / pt + 1) * cfg.q_heads * (cfg.head_dim * 4 + 8);
    }
  auto fits = [&](int64_t slots, int64_t scratch) {
    return workgroups() <= slots && c.bytes <= scratch && c.bytes + decode_bytes <= kFinerPrefillScratch;
  };
  if (f32) {
    for (c.part = kF32PrefillPart; c.part < kDefaultChunkPartition; c.part += 64) {
      c.split_keys = c.part * 3 / 2;
      if (fits(kPrefillSlots, kF32PrefillScratch)) return c;
    }
    c.split_keys = kPrefillSplitKeys;
  } else {
    c.part = kSmallPrefillPart;
    if (fits(kSmallPrefill, kSmallPrefillScratch)) return c;
  }
  c.part = std::max<int64_t>((keys / kPrefillSlots + 63) / 64 * 64, kDefaultChunkPartition);
  while (workgroups() > kPrefillSlots && c.part < longest * bs) c.part += (c.part / 8 + 63) / 64 * 64;
  return c;
}

}  // namespace

extern "C" {

int le_plan_step(const le_step_slice* slices, int n_slices, const le_plan_config* cfg_in,
                 void* host_buf, int64_t host_cap, le_step_plan* plan) {
  if (!plan || !cfg_in || n_slices < 0 || (n_slices > 0 && !slices)) return LE_EINVAL;
  le_plan_config cfg = *cfg_in;
  if (cfg.block_size <= 0 || cfg.q_heads <= 0 || cfg.kv_heads <= 0 || cfg.head_dim <= 0)
    return LE_EINVAL;
  if (cfg.kv_dtype != LE_F32 && cfg.kv_dtype != LE_BF16 && cfg.kv_dtype != LE_F16) return LE_EINVAL;
  if ((cfg.flags & ~(LE_PLAN_TWO_LAUNCHES | LE_PLAN_XCD_LOCAL)) != 0 || cfg.table_capacity < 0)
    return LE_EINVAL;
  // Fixed layout (table_capacity > 0): decode rows only, a given partition.
  const bool fixed = cfg.table_capacity > 0;
  if (fixed && cfg.partition_tokens <= 0) return LE_EINVAL;
  const int bs = cfg.block_size;
  const le_plan_config asked = cfg;
  if (cfg.chunk_q_tile <= 0) cfg.chunk_q_tile = kDefaultChunkTile;
  // 384 keys: one LDS stage of a 16-bit cache, three of fp32 at head_dim 64
  // (config 3 with fp32 K/V, 24 layers: 1.18 ms per step, against 1.62 with
  // 128-key partitions, 1.47 with 256 and 1.39 with 512)
  if (cfg.chunk_partition_tokens <= 0)
    cfg.chunk_partition_tokens = kDefaultChunkPartition;
  if (cfg.chunk_q_tile != 16 && cfg.chunk_q_tile != 32) return LE_EUNSUPPORTED;  // MFMA row tiles
  // ---- sizes, and validation of every slice against its table ----
  int64_t n_tok = 0, n_table = 0;
  int n_logits = 0, n_seqs = 0, max_pos = 0;
  std::unordered_map<int64_t, int> seq_index;
  seq_index.reserve(static_cast<size_t>(n_slices));
  std::vector<int> slice_seq(static_cast<size_t>(n_slices));
  std::vector<int> seq_first_slice;
  seq_first_slice.reserve(static_cast<size_t>(n_slices));
  for (int i = 0; i < n_slices; i++) {
    const le_step_slice& s = slices[i];
    if (s.len <= 0 || s.start < 0 || s.num_blocks < 0 || !s.tokens) return LE_EINVAL;
    if (fixed && s.len != 1) return LE_EUNSUPPORTED;
    if (fixed && s.num_blocks > cfg.table_capacity) return LE_EINVAL;
    if (s.num_blocks > 0 && !s.blocks) return LE_EINVAL;
    const int last = s.start + s.len - 1;
    if (last / bs >= s.num_blocks) return LE_EINVAL;  // a position without a block
    auto it = seq_index.find(s.seq_key);
    if (it == seq_index.end()) {
      seq_index.emplace(s.seq_key, n_seqs);
      slice_seq[i] = n_seqs++;
      seq_first_slice.push_back(i);
      n_table += s.num_blocks;
    } else {
      // Slots and block ids come from the sequence's first slice (one table
      // per sequence, as one Sequence object holds it): every later slice of
      // the key must fit that table.
      const le_step_slice& f = slices[seq_first_slice[it->second]];
      if (last / bs >= f.num_blocks) return LE_EINVAL;
      slice_seq[i] = it->second;
    }
    n_tok += s.len;
    if (s.needs_logits) n_logits++;
    max_pos = std::max(max_pos, last);
  }
  if (n_tok > INT32_MAX / 2) return LE_EUNSUPPORTED;
  // ---- decode partitions ----
  const bool auto_part = !fixed && cfg.partition_tokens <= 0;
  bool chunk_rows = false;
  for (int i = 0; i < n_slices; i++) chunk_rows |= slices[i].len > 1;
  const int max_parts = std::max(1, kMaxMergeEntries / std::max(1, cfg.q_heads / cfg.kv_heads));
  auto items_at = [&](int64_t pt) {  // decode items per kv head with partitions of pt keys
    const int64_t pb = (pt + bs - 1) / bs;
    int64_t n = 0;
    for (int i = 0; i < n_slices; i++)
      if (slices[i].len == 1) n += std::min<int64_t>((slices[i].start / bs + 1 + pb - 1) / pb, max_parts);
    return n;
  };
  int64_t part = cfg.partition_tokens, shared = 0;  // shared: one workgroup's share of the step's keys
  if (auto_part) {
    // Size decode partitions so the step has about kTargetItems workgroups,
    // two per CU. Each workgroup pays a fixed chain of dependent memory
    // round trips (block ids, then K/V; partial store, arrival counter, merge)
    // of several microseconds, so on MI355X a few long partitions stream
    // faster than many short ones (measured: 64 x 4096 rows, 2048-token
    // partitions 4.1 TB/s, 256-token 2.2 TB/s; config 2, 640-768 tokens
    // 16.3 us, 1024 17.1 us, 512 18.0 us).
    int64_t ctx = 0;
    for (int i = 0; i < n_slices; i++)
      if (slices[i].len == 1)
        for (int r = 0; r < slices[i].len; r++) ctx += slices[i].start + r + 1;
    const int64_t per_kvh = std::max<int64_t>(1, kTargetItems / cfg.kv_heads);
    shared = (ctx + per_kvh - 1) / per_kvh;
    shared = (shared + kPartitionQuantum - 1) / kPartitionQuantum * kPartitionQuantum;
    part = std::max<int64_t>(shared, kDefaultPartition);
    if (chunk_rows) {
      // In a mixed step the chunk workgroups hold most CUs for the first half
      // of the launch; splitting the decode rows further only adds merges
      // (config 3 on 32-row tiles: 22.7 us with the rule above, 22.4 us with
      // 2048 tokens).
      part = std::max<int64_t>(part, kMixedStepPartition);
    } else {
      // The rows' partitions are whole ceilings, so the rule above can
      // overshoot: grow the partition until the step's workgroups fit one
      // round at two per CU (TinyLlama-shaped decode steps, 64 rows, 4 kv
      // heads: 136-144 items per kv head ran 20.6-21.5 us per launch, 120
      // items 15-16 us).
      while (part < kMaxAutoPartition && items_at(part) * cfg.kv_heads > kTargetItems) part += kPartitionQuantum;
    }
    part = std::min<int64_t>(part, kMaxAutoPartition);
  }
  // The plain cut: these decode partitions, chunk rows over 384 keys. A step
  // that it does not split may be run without a workspace. The finer cuts
  // below pay off on such steps too (us a call, whole and split: 17 fp32 decode
  // rows of up to 640 keys, 28/4 heads x 128, 33.0 and 18.5; 4 decode rows of up
  // to 2000 keys beside 3 x 17 chunk rows, 32/8 x 128, 33.9 and 22.1; an fp32
  // prompt of 341 rows, 14/2 x 64, 27.7 and 19.6), so the plan splits them and
  // says that without a workspace its rows and tiles may run whole.
  bool splits = false;
  for (int i = 0; i < n_slices; i++)
    splits |= (slices[i].start + slices[i].len - 1) / bs + 1 >
              round_to_blocks(slices[i].len > 1 ? kDefaultChunkPartition : static_cast<int>(part), bs);
  const PrefillCut pre = cut_prefill(asked, slices, n_slices, n_tok);
  if (auto_part) {
    if (chunk_rows && pre.on && pre.bytes <= kFinerPrefillScratch) {
      // Beside prefill tiles, whose workgroups share a CU with the decode
      // rows', 1024 keys: 2 x 512 rows after 1024 keys and 32 decode rows 25.6
      // against 31.1 us. Those partitions need at most 5 MB more of partials
      // than 2048-key ones: where the tiles' own leave that much of the static
      // scratch, else 2048 as before.
      part = std::min<int64_t>(std::max<int64_t>(shared, kMixedPrefillPartition), kMaxAutoPartition);
    } else if (!chunk_rows && cfg.kv_dtype == LE_F32) {
      // fp32 keys are twice the bytes: a step that leaves CUs without a
      // workgroup takes shorter partitions, the shortest (two 32-key tiles a
      // wave on) that still gives every workgroup a CU of its own, where the
      // stream of a partition is the longest part (us a call, 640-key
      // partitions and these: 48 rows of 32-2048 keys, 14/2 heads x 64, 16.9
      // and 11.9; one row of 2000 14.3 and 10.8). A second workgroup on a CU
      // slows the first: 64 rows of 64-4096, 256 against 328 workgroups, 19.3
      // and 22.4.
      for (int64_t pt = kSmallStepPartF32; pt < part; pt += kPartitionQuantum)
        if (items_at(pt) * cfg.kv_heads <= kTargetItems / 2) {
          part = pt;
          break;
        }
    }
    cfg.partition_tokens = static_cast<int32_t>(part);
  }
  const int dec_pb = round_to_blocks(cfg.partition_tokens, bs);
  const int chk_pb = round_to_blocks(cfg.chunk_partition_tokens, bs);
  const bool mfma_chunks = true;  // chunk rows on MFMA tiles, every cache type

  // Fixed layout: every row owns parts_cap partial slots and every table
  // table_capacity entries, whatever its current length.
  const int parts_cap = fixed ? std::min((cfg.table_capacity + dec_pb - 1) / dec_pb, max_parts) : 0;
  if (fixed) n_table = static_cast<int64_t>(n_seqs) * cfg.table_capacity;

  // Table offset of each distinct sequence in the concatenated tables.
  std::vector<int32_t> seq_table_off(static_cast<size_t>(n_seqs));
  {
    int32_t o = 0;
    for (int s = 0; s < n_seqs; s++) {
      seq_table_off[s] = o;
      o += fixed ? cfg.table_capacity : slices[seq_first_slice[s]].num_blocks;
    }
  }

  // ---- work lists ----
  std::vector<le::DecodeItem> dec;
  std::vector<le::ChunkItem> chk;
  int32_t parts = 0;
  {
    int32_t t = 0;
    for (int i = 0; i < n_slices; i++) {
      const le_step_slice& s = slices[i];
      if (s.len > 1 && mfma_chunks) {
        const int rows = pre.on ? pre.rows : cfg.chunk_q_tile;
        for (int q0 = 0; q0 < s.len; q0 += rows) {
          const int nq = std::min(rows, s.len - q0);
          const int last = s.start + q0 + nq - 1;
          const int nb = last / bs + 1;
          // Long contexts get longer partitions rather than more of them.
          const int pb = std::max(chk_pb, (nb + kMaxChunkParts - 1) / kMaxChunkParts);
          if (pb > kMaxChunkItemBlocks) return LE_EUNSUPPORTED;  // the kernel stages an item's ids in LDS
          const int J = pre.on ? pre.parts(nb, bs) : (nb + pb - 1) / pb;
          const int base = J > 1 ? parts : -1;
          for (int j = 0; j < J; j++) {
            le::ChunkItem c{};
            c.tok_begin = t + q0;
            c.n_q = nq;
            c.blk_begin = static_cast<int32_t>(static_cast<int64_t>(j) * nb / J);
            c.blk_end = static_cast<int32_t>(static_cast<int64_t>(j + 1) * nb / J);
            c.part0 = J > 1 ? base + j : -1;
            c.part_stride = J;
            c.seq = slice_seq[i];
            c.part = j;
            c.key_live = std::min((c.blk_end - c.blk_begin) * bs, last + 1 - c.blk_begin * bs);
            chk.push_back(c);
          }
          if (J > 1) parts += nq * J;
        }
      } else {
        for (int r = 0; r < s.len; r++) {
          const int pos = s.start + r;
          const int nb = pos / bs + 1;
          // Partitions per row are capped (the merging workgroup loads them all).
          const int J = std::min((nb + dec_pb - 1) / dec_pb, max_parts);
          // Split rows are merged inside the decode launch by the last
          // partition to finish, so they need no combine item.
          for (int j = 0; j < J; j++) {
            le::DecodeItem d{};
            d.token = t + r;
            d.pos = pos;
            d.table_off = seq_table_off[slice_seq[i]];
            d.blk_begin = static_cast<int32_t>(static_cast<int64_t>(j) * nb / J);
            d.blk_end = static_cast<int32_t>(static_cast<int64_t>(j + 1) * nb / J);
            const int32_t first = fixed ? (t + r) * parts_cap : parts;
            d.part = J > 1 ? first + j : -1;
            d.part_begin = first;
            d.n_parts = J;
            dec.push_back(d);
          }
          if (J > 1 && !fixed) parts += J;
        }
      }
      t += s.len;
    }
  }

  // Longest work first: workgroups start over a couple of microseconds in
  // launch order, so the items on the critical path (most keys) go first.
  // Merges do not depend on the order (partials are addressed by index).
  if (fixed) parts = static_cast<int32_t>(n_tok) * parts_cap;
  // (With the XCD placement, the bins are dealt longest group first instead:
  // a row's partitions must stay adjacent until they are placed.)
  const bool xcd_local = (cfg.flags & LE_PLAN_XCD_LOCAL) && !fixed;
  bool dec_split = false;
  for (const auto& d : dec) dec_split |= d.part >= 0;
  if (xcd_local && dec_split) {
    dec = place_decode_items(dec);
  } else {
    std::stable_sort(dec.begin(), dec.end(), [](const le::DecodeItem& a, const le::DecodeItem& b) {
      return a.blk_end - a.blk_begin > b.blk_end - b.blk_begin;
    });
  }
  bool chunk_split = false;
  for (const auto& c : chk) chunk_split |= c.part0 >= 0;
  // Prefill workgroups are numbered with the kv heads innermost: with a
  // multiple of 8 of them, one head's tiles share an XCD in any order.
  if (chunk_split && !(pre.on && cfg.kv_heads % kXcds == 0)) {
    chk = place_chunk_items(chk);
  } else {
    std::stable_sort(chk.begin(), chk.end(), [](const le::ChunkItem& a, const le::ChunkItem& b) {
      return a.blk_end - a.blk_begin > b.blk_end - b.blk_begin;
    });
  }

  if (fixed) {
    // one item count for every step of this row count: each row has at most
    // parts_cap partitions, so rows * parts_cap items, padded with empty
    // ones (n_parts 0: resolved as no work)
    const size_t cap_items = static_cast<size_t>(n_tok) * parts_cap;
    if (dec.size() > cap_items) return LE_EUNSUPPORTED;  // unreachable: J <= parts_cap per row
    le::DecodeItem pad{};
    pad.token = -1;
    pad.part = -1;
    dec.resize(cap_items, pad);
  }

  // ---- layout: every array 256-byte aligned in one buffer ----
  le_step_plan P{};
  P.cfg = cfg;
  if (pre.on) {
    P.cfg.chunk_q_tile = pre.wide ? le::kWidePrefillTiles : le::kPrefillTiles;
    P.cfg.chunk_partition_tokens = 0;
  }
  if (!fixed && !splits && parts > 0 && (pre.on || chk.empty())) P.cfg.chunk_partition_tokens = le::kMayRunWhole;
  P.n_tokens = static_cast<int32_t>(n_tok);
  P.n_seqs = n_seqs;
  P.n_table = static_cast<int32_t>(n_table);
  P.n_logits = n_logits;
  P.n_decode_items = static_cast<int32_t>(dec.size());
  P.n_chunk_items = static_cast<int32_t>(chk.size());
  P.n_combine_items = 0;  // chunk rows merge inside their launch
  P.n_parts = parts;
  P.max_pos = max_pos;
  P.n_slices = n_slices;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    const int64_t o = off;
    off = align256(off + std::max<int64_t>(bytes, 4));
    return o;
  };
  P.off_token_ids = take(n_tok * 4);
  P.off_positions = take(n_tok * 4);
  P.off_slots = take(n_tok * 4);
  P.off_token_seq = take(n_tok * 4);
  P.off_tables = take(n_table * 4);
  P.off_table_offset = take(static_cast<int64_t>(n_seqs) * 4);
  P.off_cu_seqlens_q = take(static_cast<int64_t>(n_slices + 1) * 4);
  P.off_seq_lens_k = take(static_cast<int64_t>(n_slices) * 4);
  P.off_logit_rows = take(static_cast<int64_t>(n_logits) * 4);
  P.off_decode_items = take(static_cast<int64_t>(dec.size()) * sizeof(le::DecodeItem));
  P.off_chunk_items = take(static_cast<int64_t>(chk.size()) * sizeof(le::ChunkItem));
  P.off_combine_items = take(0);
  // Each work item's block ids at a fixed stride (decode items, then chunk
  // items), so a workgroup can fetch them in the same memory round trip as
  // its item. A prefill tile may hold the whole of a long context and would
  // widen every item's row, past what a decode workgroup takes ahead of its
  // item (64 rows of 1024 keys beside a chunk after 16384, block size 8: 128 ids
  // against 2304): one with more ids than the decode items and kTileListIds
  // reads the step's tables instead (seq: ~ where its table starts), which
  // costs it nothing, as its loads wait for the item anyway.
  int32_t ids_stride = 0;
  for (const auto& d : dec) ids_stride = std::max(ids_stride, d.blk_end - d.blk_begin);
  const int32_t listed = std::max(ids_stride, kTileListIds);
  for (auto& c : chk) {
    if (pre.on && c.blk_end - c.blk_begin > listed) c.seq = ~seq_table_off[c.seq];
    else ids_stride = std::max(ids_stride, c.blk_end - c.blk_begin);
  }
  if (fixed) ids_stride = std::max(dec_pb, (cfg.table_capacity + parts_cap - 1) / parts_cap);
  ids_stride = (ids_stride + 3) / 4 * 4;
  P.decode_ids_stride = ids_stride;
  P.xcd_local = xcd_local ? 1 : 0;
  P.off_decode_ids = take(static_cast<int64_t>(dec.size() + chk.size()) * ids_stride * 4);
  P.bytes = off;
  P.dev = nullptr;
  if (!host_buf || host_cap < P.bytes) {
    *plan = P;
    return LE_ENOSPACE;
  }

  char* base = static_cast<char*>(host_buf);
  auto arr = [&](int64_t o) { return reinterpret_cast<int32_t*>(base + o); };
  int32_t* token_ids = arr(P.off_token_ids);
  int32_t* positions = arr(P.off_positions);
  int32_t* slots = arr(P.off_slots);
  int32_t* token_seq = arr(P.off_token_seq);
  int32_t* tables = arr(P.off_tables);
  int32_t* table_offset = arr(P.off_table_offset);
  int32_t* cu_q = arr(P.off_cu_seqlens_q);
  int32_t* lens_k = arr(P.off_seq_lens_k);
  int32_t* logit_rows = arr(P.off_logit_rows);

  int32_t nt = 0;
  for (int s = 0; s < n_seqs; s++) {
    const le_step_slice& f = slices[seq_first_slice[s]];
    table_offset[s] = nt;
    if (f.num_blocks) std::memcpy(tables + nt, f.blocks, sizeof(int32_t) * f.num_blocks);
    const int32_t width = fixed ? cfg.table_capacity : f.num_blocks;
    for (int32_t j = f.num_blocks; j < width; j++) tables[nt + j] = -1;
    nt += width;
  }
  int32_t t = 0, r = 0;
  cu_q[0] = 0;
  for (int i = 0; i < n_slices; i++) {
    const le_step_slice& s = slices[i];
    // Slots come from the table of the sequence (its first slice), as the
    // reference reads them from the Sequence object.
    const le_step_slice& f = slices[seq_first_slice[slice_seq[i]]];
    for (int k = 0; k < s.len; k++) {
      const int pos = s.start + k;
      token_ids[t] = s.tokens[pos];
      positions[t] = pos;
      token_seq[t] = slice_seq[i];
      slots[t] = static_cast<int32_t>(static_cast<int64_t>(f.blocks[pos / bs]) * bs + pos % bs);
      t++;
    }
    if (s.needs_logits) logit_rows[r++] = t - 1;
    cu_q[i + 1] = t;
    lens_k[i] = s.start + s.len;
  }
  if (!dec.empty()) {
    std::memcpy(base + P.off_decode_items, dec.data(), dec.size() * sizeof(le::DecodeItem));
    int32_t* ids = arr(P.off_decode_ids);
    for (size_t k = 0; k < dec.size(); k++) {
      const le::DecodeItem& d = dec[k];
      int32_t* row = ids + k * static_cast<size_t>(ids_stride);
      for (int j = 0; j < ids_stride; j++)
        row[j] = j < d.blk_end - d.blk_begin ? tables[d.table_off + d.blk_begin + j] : -1;
    }
  }
  if (!chk.empty()) {
    std::memcpy(base + P.off_chunk_items, chk.data(), chk.size() * sizeof(le::ChunkItem));
    int32_t* ids = arr(P.off_decode_ids) + dec.size() * static_cast<size_t>(ids_stride);
    for (size_t k = 0; k < chk.size(); k++) {
      const le::ChunkItem& c = chk[k];
      const int n = c.seq < 0 ? 0 : c.blk_end - c.blk_begin;
      const int32_t* from = tables + (c.seq < 0 ? 0 : table_offset[c.seq]) + c.blk_begin;
      int32_t* row = ids + k * static_cast<size_t>(ids_stride);
      for (int j = 0; j < ids_stride; j++) row[j] = j < n ? from[j] : -1;
    }
  }
  *plan = P;
  return LE_OK;
}

int le_plan_upload(le_step_plan* plan, const void* host_buf, void* dev_buf, hipStream_t stream) {
  if (!plan || !host_buf || !dev_buf || plan->bytes <= 0) return LE_EINVAL;
  const hipError_t e = hipMemcpyAsync(dev_buf, host_buf, static_cast<size_t>(plan->bytes),
                                      hipMemcpyHostToDevice, stream);
  if (e != hipSuccess) return static_cast<int>(e);
  plan->dev = dev_buf;
  return LE_OK;
}

}  // extern "C"
