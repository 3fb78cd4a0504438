// Ragged paged attention of a mixed step in one launch (hot-path part 3):
// the step's prefill-chunk rows (chunk_wg, attention_chunk_wg.h) and decode
// rows (decode_wg, attention_decode_wg.h) as workgroups of one grid.
//
// With two launches the chunk rows' latency-bound phases (stage, compute,
// partial store, merge) and the decode rows' HBM streaming run one after the
// other, with a launch gap between them. In one grid the decode workgroups
// stream on the CUs the chunk workgroups leave free, and start on the others
// as chunk workgroups retire. Chunk workgroups come first in the grid: theirs
// is the longer dependent chain (a split tile's merge waits for its last
// partition).
//
// Both kinds keep their own merges inside the launch: partition indices and
// arrival counters are disjoint between them (the plan numbers partitions
// across both lists; counters are indexed by a row's or tile's first token).
// Beside 32-row tiles (ragged_kernel) workgroups are 512 threads (the chunk
// workgroup's eight waves) and the decode workgroups run as eight waves as well;
// beside prefill tiles, what a step takes by default, both are 256 threads. The LDS is the larger of the two.
#include "attention_chunk_wg.h"
#include "attention_decode_wg.h"
#include "attention_prefill_f32_wg.h"
#include "llm_engine_amd.h"

namespace le {
namespace {

constexpr int kRaggedThreads = chk::kThreads;
constexpr int kDecodeWaves = kRaggedThreads / kWave;

template <typename KV, int HD> union RaggedSmem {
  chk::ChunkSmem<KV, HD> c;
  dec::DecodeSmem<KV, HD, kDecodeWaves> d;
};

template <typename ACT, typename KV, int HD>
__global__ __launch_bounds__(kRaggedThreads) void ragged_kernel(DecodeParams dp, ChunkParams cp) {
  __shared__ RaggedSmem<KV, HD> sm;
  const int n_chunk_wg = cp.n_items * cp.kv_heads;
  const int b = blockIdx.x;
  if (b < n_chunk_wg) {
    // item-major within each kv head, as the chunk kernel's 2-D grid (the
    // plan places a split tile's partitions at item indices equal modulo 8)
    chk::chunk_wg<ACT, KV, HD>(cp, sm.c, b % cp.n_items, b / cp.n_items);
  } else {
    // item-major within each kv head, as the decode kernel's 2-D grid: the
    // plan places a split row's partitions at item indices equal modulo 8,
    // so they share an XCD in either launch
    const int d = b - n_chunk_wg;
    dec::decode_wg<ACT, KV, HD, kDecodeWaves>(dp, sm.d, d % dp.n_rows, d / dp.n_rows, 0);
  }
}

// The same for chunk rows cut into prefill tiles of a 16-bit cache: 256-thread
// workgroups of both kinds, two of any per CU. Bound like the prefill kernel
// in steps with large chunks, by the decode rows' streaming and the tiles'
// serial chain in small ones. Against the kernel above (us per call): 2 x 512
// rows after 1024 keys and 32 decode rows of 256-2048, 14/2 heads x 64, 28.9
// and 25.6; 8 x 512 after 4096, 32/4 x 64, 369 and 171; one chunk of 64 after
// nothing, 16.2 and 11.6; 8/8 x 128 and 8 x 512 after 1024, 321 and 80.
template <typename KV, int HD> union RaggedPrefillSmem {
  pre::PrefillSmem<HD> c;
  dec::DecodeSmem<KV, HD, pre::kWaves> d;
};

// kWhole: without a workspace, split rows and tiles run whole (instantiations of
// their own, so that the usual launch is not shaped by it).
template <typename ACT, typename KV, int HD, int NC, bool kWhole>
__global__ __launch_bounds__(pre::kThreads, 2) void ragged_prefill_kernel(DecodeParams dp, ChunkParams cp) {
  __shared__ RaggedPrefillSmem<KV, HD> sm;
  const int n_chunk_wg = cp.n_items * cp.kv_heads;
  const int b = blockIdx.x;
  if (b < n_chunk_wg) {
    pre::prefill_wg<ACT, KV, HD, NC, kWhole>(cp, sm.c, b / cp.kv_heads, b % cp.kv_heads);
  } else {
    const int d = b - n_chunk_wg;
    dec::decode_wg<ACT, KV, HD, pre::kWaves, false, kWhole>(dp, sm.d, d % dp.n_rows, d / dp.n_rows, 0);
  }
}

// And for fp32 caches of head_dim 64. Bound as above: 64 decode rows of 2048
// keys beside one chunk of 16, 14/2 heads, 37.1 us on the kernel above and 33.2
// here; 32 decode rows and 2 x 512 rows after 0-1024, 48.6 and 44.9.
template <int HD> union RaggedPrefillF32Smem {
  pre::PrefillF32Smem<HD> c;
  dec::DecodeSmem<float, HD, pre::kWaves> d;
};

template <typename ACT, int HD, bool kWhole>
__global__ __launch_bounds__(pre::kThreads, 2) void ragged_prefill_f32_kernel(DecodeParams dp, ChunkParams cp) {
  __shared__ RaggedPrefillF32Smem<HD> sm;
  const int n_chunk_wg = cp.n_items * cp.kv_heads;
  const int b = blockIdx.x;
  if (b < n_chunk_wg) {
    pre::prefill_f32_wg<ACT, HD, kWhole>(cp, sm.c, b / cp.kv_heads, b % cp.kv_heads);
  } else {
    const int d = b - n_chunk_wg;
    dec::decode_wg<ACT, float, HD, pre::kWaves, false, kWhole>(dp, sm.d, d % dp.n_rows, d / dp.n_rows, 0);
  }
}

}  // namespace

namespace {

template <bool kWhole>
hipError_t launch_prefill(const DecodeParams& d, const ChunkParams& c, bool wide, int act_dtype, int kv_dtype,
                          const dim3& grid, hipStream_t s) {
  return with_dtype(act_dtype, [&](auto a) {
    if (kv_dtype == LE_F32) {
      if (c.head_dim != 64 || wide) return hipErrorInvalidValue;
      ragged_prefill_f32_kernel<decltype(a), 64, kWhole><<<grid, pre::kThreads, 0, s>>>(d, c);
      return hipGetLastError();
    }
    return with_dtype16(kv_dtype, [&](auto k) {
      using ACT = decltype(a);
      using KV = decltype(k);
      if (c.head_dim == 128) ragged_prefill_kernel<ACT, KV, 128, 1, kWhole><<<grid, pre::kThreads, 0, s>>>(d, c);
      else if (wide) ragged_prefill_kernel<ACT, KV, 64, 2, kWhole><<<grid, pre::kThreads, 0, s>>>(d, c);
      else ragged_prefill_kernel<ACT, KV, 64, 1, kWhole><<<grid, pre::kThreads, 0, s>>>(d, c);
      return hipGetLastError();
    });
  });
}

}  // namespace

hipError_t attention_ragged_prefill(const DecodeParams& d, const ChunkParams& c, bool wide, int act_dtype,
                                    int kv_dtype, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(c.n_items + d.n_rows) * c.kv_heads;
  if (n <= 0) return hipSuccess;
  if (n > 0x7fffffff || d.kv_heads != c.kv_heads || d.head_dim != c.head_dim || !d.items ||
      (d.item_ids == nullptr) != (c.item_ids == nullptr) || (wide && c.head_dim != 64))
    return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(n));
  return d.item_ids ? launch_prefill<false>(d, c, wide, act_dtype, kv_dtype, grid, s)
                    : launch_prefill<true>(d, c, wide, act_dtype, kv_dtype, grid, s);
}

hipError_t attention_ragged(const DecodeParams& d, const ChunkParams& c, int act_dtype, int kv_dtype,
                            hipStream_t s) {
  const int64_t n = static_cast<int64_t>(c.n_items + d.n_rows) * c.kv_heads;
  if (n <= 0) return hipSuccess;
  if (n > 0x7fffffff || d.kv_heads != c.kv_heads || d.head_dim != c.head_dim || !d.items)
    return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(n));
  return with_dtype(act_dtype, [&](auto a) {
    return with_dtype(kv_dtype, [&](auto k) {
      using ACT = decltype(a);
      using KV = decltype(k);
      if (c.head_dim == 64) ragged_kernel<ACT, KV, 64><<<grid, kRaggedThreads, 0, s>>>(d, c);
      else ragged_kernel<ACT, KV, 128><<<grid, kRaggedThreads, 0, s>>>(d, c);
      return hipGetLastError();
    });
  });
}

}  // namespace le

#ifdef LE_TIMING
// Measurement builds only: the mixed-step kernel's phase stamps of its last
// launch (decode and chunk workgroups; slot 7 tells them apart).
extern "C" int le_timing_read_ragged(void* host, int64_t bytes) {
  return static_cast<int>(hipMemcpyFromSymbol(host, HIP_SYMBOL(le::g_timing), static_cast<size_t>(bytes), 0,
                                              hipMemcpyDeviceToHost));
}
#endif
