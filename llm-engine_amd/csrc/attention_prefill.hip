// Prefill chunk rows (hot-path part 3): the kernels over prefill tiles. The
// workgroups are prefill_wg (16-bit caches, attention_prefill_wg.h) and
// prefill_f32_wg (fp32, attention_prefill_f32_wg.h), which the mixed-step
// kernels (attention_ragged.hip) share.
#include "attention_prefill_f32_wg.h"
#include "llm_engine_amd.h"

namespace le {
namespace {

template <typename ACT, typename KV, int HD, int NC>
__global__ __launch_bounds__(pre::kThreads, 2) void prefill_kernel(ChunkParams p) {
  __shared__ pre::PrefillSmem<HD> sm;
  // kv heads innermost: with 8 (4, 2) of them an XCD serves one (of one, of
  // two) head's K/V, whose rows its L2 then holds for all tiles of a sequence
  pre::prefill_wg<ACT, KV, HD, NC, true>(p, sm, blockIdx.x / p.kv_heads, blockIdx.x % p.kv_heads);
}

template <typename ACT, int HD>
__global__ __launch_bounds__(pre::kThreads, 2) void prefill_f32_kernel(ChunkParams p) {
  __shared__ pre::PrefillF32Smem<HD> sm;
  pre::prefill_f32_wg<ACT, HD, true>(p, sm, blockIdx.x / p.kv_heads, blockIdx.x % p.kv_heads);
}

}  // namespace

hipError_t attention_prefill(const ChunkParams& p, bool wide, int act_dtype, int kv_dtype, hipStream_t s) {
  if (p.n_items <= 0) return hipSuccess;
  if (static_cast<int64_t>(p.n_items) * p.kv_heads > 0x7fffffff || (wide && p.head_dim != 64)) return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(p.n_items * p.kv_heads));
  return with_dtype(act_dtype, [&](auto a) {
    if (kv_dtype == LE_F32) {
      if (p.head_dim != 64 || wide) return hipErrorInvalidValue;
      prefill_f32_kernel<decltype(a), 64><<<grid, pre::kThreads, 0, s>>>(p);
      return hipGetLastError();
    }
    return with_dtype16(kv_dtype, [&](auto k) {
      using ACT = decltype(a);
      using KV = decltype(k);
      if (p.head_dim == 128) prefill_kernel<ACT, KV, 128, 1><<<grid, pre::kThreads, 0, s>>>(p);
      else if (wide) prefill_kernel<ACT, KV, 64, 2><<<grid, pre::kThreads, 0, s>>>(p);
      else prefill_kernel<ACT, KV, 64, 1><<<grid, pre::kThreads, 0, s>>>(p);
      return hipGetLastError();
    });
  });
}

}  // namespace le
