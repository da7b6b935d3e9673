// Prefill attention: kernel and host launcher. What bounds the work and how
// it is laid out: attention_prefill.h.

#include <c10/hip/HIPStream.h>

#include "attention.h"

namespace vllm_amd {

template <typename Tag, typename CTag, int HD>
__global__ __launch_bounds__(PF_BLOCK, pf_per_cu<HD>)
void prefill_attention_kernel(const PrefillArgs<CTag> a,
                              const int num_decodes) {
  __shared__ __align__(16) char lds[pf_lds<HD>];
  // One XCD takes every eighth workgroup, so with the KV head fastest a
  // head's tiles stay in one L2. Late tiles attend most keys: first.
  prefill_tile<Tag, CTag, HD>(a, blockIdx.x, num_decodes + blockIdx.z,
                              blockIdx.y, lds);
}

void check_prefill(const torch::Tensor& out, const torch::Tensor& q,
                   const torch::Tensor& kv_cache) {
  const int num_q_heads = q.size(1);
  const int head_dim = q.size(2);
  const int num_kv_heads = kv_cache.size(2);
  TORCH_CHECK(head_dim == 64 || head_dim == 128 || head_dim == 256,
              "prefill kernel supports head_dim 64/128/256");
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == head_dim &&
              q.stride(0) % 8 == 0, "q must be head-contiguous [T,H,D]");
  TORCH_CHECK(out.is_contiguous(), "out must be contiguous");
  TORCH_CHECK(kv_cache.size(3) == KVTILE, "cache block_size must be 64");
  TORCH_CHECK(num_q_heads % num_kv_heads == 0);
}

// ---------------------------------------------------------------------------
// Host launcher. q/out: [T, Hq, D] covering the WHOLE step batch;
// rows for prefill requests are query_start_loc[num_decodes..num_reqs].
void prefill_attention(torch::Tensor out, torch::Tensor q,
                       torch::Tensor kv_cache, torch::Tensor block_table,
                       torch::Tensor query_start_loc, torch::Tensor seq_lens,
                       double scale, int64_t num_decodes,
                       int64_t max_query_len, int64_t sliding_window) {
  const int num_reqs = seq_lens.size(0);
  const int num_prefills = num_reqs - (int)num_decodes;
  if (num_prefills == 0) return;
  check_prefill(out, q, kv_cache);
  const int head_dim = q.size(2);
  const int num_kv_heads = kv_cache.size(2);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  dim3 grid(num_kv_heads,
            prefill_tiles(max_query_len, (int)q.size(1) / num_kv_heads),
            num_prefills);
  const bool fp8c = kv_cache.scalar_type() == torch::kFloat8_e4m3fn;
  auto launch = [&](auto tag, auto ctag, auto dim) {
    using CTag = decltype(ctag);
    hipLaunchKernelGGL(
        (prefill_attention_kernel<decltype(tag), CTag, decltype(dim)::value>),
        grid, dim3(PF_BLOCK), 0, stream,
        prefill_args<CTag>(out, q, kv_cache, block_table, query_start_loc,
                           seq_lens, scale, sliding_window),
        (int)num_decodes);
  };
  auto dispatch = [&](auto dim) {
    if (q.scalar_type() == torch::kBFloat16) {
      if (fp8c) launch(BF16Tag{}, FP8CacheTag{}, dim);
      else      launch(BF16Tag{}, BF16Tag{}, dim);
    } else {
      if (fp8c) launch(FP16Tag{}, FP8CacheTag{}, dim);
      else      launch(FP16Tag{}, FP16Tag{}, dim);
    }
  };
  if (head_dim == 64) dispatch(std::integral_constant<int, 64>{});
  else if (head_dim == 128) dispatch(std::integral_constant<int, 128>{});
  else dispatch(std::integral_constant<int, 256>{});
  HIP_CHECK_KERNEL();
}

}  // namespace vllm_amd
