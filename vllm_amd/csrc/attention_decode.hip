// Paged decode attention: kernel and host launcher. What bounds the work and
// how it is laid out: attention_decode.h.

#include <c10/hip/HIPStream.h>

#include "attention.h"

namespace vllm_amd {

template <typename Tag, typename CTag, bool WHOLE, int HD, int WPR>
__global__ __launch_bounds__(DEC_BLOCK, 2) void paged_decode_kernel(
    const DecodeArgs<CTag> a) {
  __shared__ __align__(16) char lds[dec_lds<CTag, HD>];
  decode_rows<Tag, CTag, WHOLE, HD, WPR>(a, blockIdx.x, blockIdx.y,
                                         blockIdx.z, lds);
}

// Rows of a few steps leave three of a workgroup's four waves idle, and
// starting and merging it costs more than its keys: from half the waves
// that run at a time on, each takes a row of at most 128 keys of its own;
// of up to 512 (the least that a captured step is told) where rows fill
// the chip twice over. us, workgroup / wave a row, 32/8 heads of 128: 1024
// rows x 1..32 keys 49 / 20, 33..64 56 / 35, 129..176 125 / 121, 512 377 /
// 378; 128 x 1..128 11.1 / 9.3; 64 x 128 7.6 / 8.8, 512 x 1..512 104 / 106.
// Heads of 256: 512 x 128 97.6 / 99.3, 1..128 49 / 45, 1..512 195 / 207.
bool decode_waves(int64_t units, int64_t head_dim, int64_t num_parts,
                  int64_t span) {
  return num_parts == 1 &&
         ((span <= 128 && units >= (head_dim == 64 ? 1536 : 1024)) ||
          (span <= 512 && units >= 4096 && head_dim <= 128));
}

// Checks the operands of num_seqs decode rows and lays them out.
DecodePlan plan_decode(const torch::Tensor& out, const torch::Tensor& q,
                       const torch::Tensor& kv_cache, int num_seqs,
                       double scale, int64_t max_seq_len,
                       int64_t sliding_window, const torch::Tensor& tmp_out,
                       const torch::Tensor& tmp_lse) {
  const int num_q_heads = q.size(1);
  const int head_dim = q.size(2);
  const int num_kv_heads = kv_cache.size(2);
  const int group = num_q_heads / num_kv_heads;
  TORCH_CHECK(head_dim == 64 || head_dim == 128 || head_dim == 256,
              "decode kernel supports head_dim 64/128/256, got ", head_dim);
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == head_dim &&
              q.stride(0) % 8 == 0, "q must be head-contiguous [T,H,D]");
  TORCH_CHECK(out.is_contiguous(), "out must be contiguous");
  TORCH_CHECK(kv_cache.size(3) == 64, "cache block_size must be 64");
  TORCH_CHECK(group >= 1 && group <= MAX_GROUP && num_q_heads ==
              group * num_kv_heads, "GQA group must be 1..8, got ", group);
  int num_parts = 1;
  if (tmp_out.numel() > 0) {
    TORCH_CHECK(tmp_out.dim() == 4 && tmp_lse.dim() == 4 &&
                tmp_out.is_contiguous() && tmp_lse.is_contiguous() &&
                tmp_out.size(0) == num_seqs && tmp_lse.size(0) == num_seqs &&
                tmp_out.size(1) == num_q_heads &&
                tmp_lse.size(1) == num_q_heads &&
                tmp_out.size(2) == tmp_lse.size(2) &&
                tmp_out.size(3) == head_dim && tmp_lse.size(3) == 2,
                "decode scratch must be [T, Hq, parts, D] and "
                "[T, Hq, parts, 2]");
    num_parts = std::min((int)tmp_out.size(2), MAX_PARTS);
  }
  // A window starts on a multiple of 32 keys, up to 31 before it.
  int64_t span = std::max<int64_t>(max_seq_len, 1);
  if (sliding_window > 0)
    span = std::min(span, sliding_window + DEC_KEYS - 1);
  const int unit = DEC_WAVES * DEC_KEYS;
  const int part_len =
      (int)((span + (int64_t)num_parts * unit - 1) /
            ((int64_t)num_parts * unit)) * unit;
  const int64_t units = (int64_t)num_seqs * num_kv_heads;
  const bool wave_rows = decode_waves(units, head_dim, num_parts, span);
  torch::Tensor arrived;
  if (num_parts > 1) arrived = arrival_counters(q, units);
  return {num_parts, part_len, wave_rows, (float)scale * DEC_LOG2E, arrived};
}

// ---------------------------------------------------------------------------
// Host launcher. q: [Tdec, Hq, D] (contiguous slice of the step's q);
// out: [Tdec, Hq, D]; kv_cache: [2, blocks, Hkv, 64, D];
// block_table/seq_lens cover the decode rows (rows 0..Tdec-1).
// tmp_out [Tdec, Hq, parts, D] and tmp_lse [Tdec, Hq, parts, 2] say into
// how many partitions a row's keys are split; empty means one.
void paged_decode_attention(torch::Tensor out, torch::Tensor q,
                            torch::Tensor kv_cache,
                            torch::Tensor block_table,
                            torch::Tensor seq_lens, double scale,
                            int64_t max_seq_len, int64_t sliding_window,
                            torch::Tensor tmp_out, torch::Tensor tmp_lse) {
  const int num_seqs = q.size(0);
  if (num_seqs == 0) return;
  const int head_dim = q.size(2);
  const DecodePlan p =
      plan_decode(out, q, kv_cache, num_seqs, scale, max_seq_len,
                  sliding_window, tmp_out, tmp_lse);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const dim3 grid((unsigned)kv_cache.size(2),
                  p.wave_rows ? ceil_div(num_seqs, DEC_WAVES) : num_seqs,
                  p.num_parts);

  auto launch = [&](auto tag, auto ctag, auto dim, auto whole, auto wpr) {
    using Tag = decltype(tag);
    using CTag = decltype(ctag);
    constexpr int HD = decltype(dim)::value;
    hipLaunchKernelGGL(
        (paged_decode_kernel<Tag, CTag, decltype(whole)::value, HD,
                             decltype(wpr)::value>),
        grid, dim3(DEC_BLOCK), 0, stream,
        decode_args<CTag>(p, out, q, kv_cache, num_seqs, block_table,
                          seq_lens, sliding_window, tmp_out, tmp_lse));
  };
  auto by_dim = [&](auto tag, auto ctag, auto whole, auto wpr) {
    if (head_dim == 64)
      launch(tag, ctag, std::integral_constant<int, 64>{}, whole, wpr);
    else if (head_dim == 128)
      launch(tag, ctag, std::integral_constant<int, 128>{}, whole, wpr);
    else
      launch(tag, ctag, std::integral_constant<int, 256>{}, whole, wpr);
  };
  const bool fp8c = kv_cache.scalar_type() == torch::kFloat8_e4m3fn;
  auto by_type = [&](auto whole, auto wpr) {
    if (q.scalar_type() == torch::kBFloat16) {
      if (fp8c) by_dim(BF16Tag{}, FP8CacheTag{}, whole, wpr);
      else      by_dim(BF16Tag{}, BF16Tag{}, whole, wpr);
    } else {
      if (fp8c) by_dim(FP16Tag{}, FP8CacheTag{}, whole, wpr);
      else      by_dim(FP16Tag{}, FP16Tag{}, whole, wpr);
    }
  };
  using one = std::integral_constant<int, 1>;
  using four = std::integral_constant<int, DEC_WAVES>;
  if (p.wave_rows)           by_type(std::true_type{}, one{});
  else if (p.num_parts == 1) by_type(std::true_type{}, four{});
  else                       by_type(std::false_type{}, four{});
  HIP_CHECK_KERNEL();
}

}  // namespace vllm_amd
