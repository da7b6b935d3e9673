// Host side that the attention launches share: checks of the operands and
// the arguments of attention_decode.h and attention_prefill.h.
#pragma once

#include <torch/all.h>

#include "attention_decode.h"
#include "attention_prefill.h"

namespace vllm_amd {

struct DecodePlan {
  int num_parts, part_len;
  bool wave_rows;   // a wave a row
  float scale_log2;
  torch::Tensor arrived;
};
DecodePlan plan_decode(const torch::Tensor& out, const torch::Tensor& q,
                       const torch::Tensor& kv_cache, int num_seqs,
                       double scale, int64_t max_seq_len,
                       int64_t sliding_window, const torch::Tensor& tmp_out,
                       const torch::Tensor& tmp_lse);

template <typename CTag>
DecodeArgs<CTag> decode_args(const DecodePlan& p, const torch::Tensor& out,
                             const torch::Tensor& q,
                             const torch::Tensor& kv_cache, int num_seqs,
                             const torch::Tensor& block_table,
                             const torch::Tensor& seq_lens,
                             int64_t sliding_window,
                             const torch::Tensor& tmp_out,
                             const torch::Tensor& tmp_lse) {
  const bool whole = p.num_parts == 1;
  const int num_kv_heads = (int)kv_cache.size(2);
  return {(short*)out.data_ptr(),
          whole ? nullptr : tmp_out.data_ptr<float>(),
          whole ? nullptr : tmp_lse.data_ptr<float>(),
          whole ? nullptr : (unsigned*)p.arrived.data_ptr<int>(),
          (const short*)q.data_ptr(),
          (const typename CacheTraits<CTag>::elem*)kv_cache.data_ptr(),
          block_table.data_ptr<int>(),
          seq_lens.data_ptr<int>(),
          p.scale_log2,
          (int)q.size(1) / num_kv_heads,
          num_kv_heads,
          num_seqs,
          (int)block_table.size(1),
          p.num_parts,
          p.part_len,
          kv_cache.stride(0),
          q.stride(0),
          (int)sliding_window};
}

void check_prefill(const torch::Tensor& out, const torch::Tensor& q,
                   const torch::Tensor& kv_cache);

template <typename CTag>
PrefillArgs<CTag> prefill_args(const torch::Tensor& out,
                               const torch::Tensor& q,
                               const torch::Tensor& kv_cache,
                               const torch::Tensor& block_table,
                               const torch::Tensor& query_start_loc,
                               const torch::Tensor& seq_lens, double scale,
                               int64_t sliding_window) {
  // The kernel takes row maxima before scaling: a negative scale moves
  // to the queries, and a scale of zero is a tiny one (all keys equal).
  const int num_kv_heads = (int)kv_cache.size(2);
  return {(short*)out.data_ptr(),
          (const short*)q.data_ptr(),
          (const typename CacheTraits<CTag>::elem*)kv_cache.data_ptr(),
          block_table.data_ptr<int>(),
          query_start_loc.data_ptr<int>(),
          seq_lens.data_ptr<int>(),
          std::max(std::fabs((float)scale * LOG2E), 1e-30f),
          (int)(scale < 0),
          (int)q.size(1) / num_kv_heads,
          num_kv_heads,
          (int)block_table.size(1),
          kv_cache.stride(0),
          q.stride(0),
          (int)sliding_window};
}

// 128-row tiles of a request of max_query_len tokens, at most.
inline int prefill_tiles(int64_t max_query_len, int group) {
  return (int)((max_query_len * group + PF_ROWS - 1) / PF_ROWS);
}

}  // namespace vllm_amd
