// Attention of a step that holds decode rows and portions of prompts, in one
// launch (gfx950). Rows are bound by HBM (attention_decode.h), portions by
// the matrix cores (attention_prefill.h): one after the other each leaves
// idle what the other wants, so their workgroups alternate over the grid and
// meet on every CU.

#include <c10/hip/HIPStream.h>

#include "attention.h"

namespace vllm_amd {

namespace {

constexpr int max_lds(int a, int b) { return a > b ? a : b; }

// Units of num_kv_heads workgroups (the KV head fastest, so that with eight
// a head's keys stay in one XCD's L2): `tiles` units are tiles of portions,
// the last of each portion first, `rows` units (row, partition) pairs. Tiles
// are spread evenly over the first `spread` units: over all where they are
// at least two of three, otherwise so that they are two of three while they
// last, as the last to start should be short.
//
// Workgroups of an XCD are dealt to its CUs four ways in turn, so work that
// comes back every second or fourth unit meets on some CUs only: one tile of
// two went to one half of them; short portions beside a long one leave units
// without work, and every fourth was a tile (portions of 2000, 100 and 100 tokens
// beside 8 x 4000 keys 129 us in turn, 147 in one launch, 91 now; 64 x 2000 with
// a window of 512 62, 86, 50). So the units are turned by one place in each
// group of four.
//
// 32/8 heads of 128, us one after the other and so: 96 rows x 100..4000
// keys and portions of 400, 700 and 1001 tokens after 0 to 4096 291 -> 208;
// 200 rows x 100..2000 and 2 of 100 and 200 tokens 152 -> 140; 16 rows x
// 100..300 and 30 of 17..200 30.7 -> 27.9; 32/4 heads, 32 rows x 2000..4000
// and 4 of 1000..2000 140 -> 124 (runs of 256 tiles and 256 rows in turn were
// a fifth slower there).
struct Mix { int tiles, rows, spread, num_prefills; };

template <typename Tag, typename CTag, bool WHOLE, int HD>
__global__ __launch_bounds__(PF_BLOCK, pf_per_cu<HD>)
void mixed_attention_kernel(
    const DecodeArgs<CTag> d, const PrefillArgs<CTag> p, const Mix mix) {
  static_assert(PF_BLOCK == DEC_BLOCK);
  __shared__ __align__(16) char lds[max_lds(pf_lds<HD>, dec_lds<CTag, HD>)];
  const int kvh = blockIdx.x;
  const auto before = [&](int n) {   // tiles among the first n units
    return (int)((int64_t)min(n, mix.spread) * mix.tiles / mix.spread);
  };
  int y = blockIdx.y;
  if (y < ((mix.tiles + mix.rows) & ~3)) y = (y & ~3) | ((y + (y >> 2)) & 3);
  const int at = before(y);
  const bool tile = before(y + 1) > at;
  const int u = tile ? at : y - at;
  if (tile)
    prefill_tile<Tag, CTag, HD>(p, kvh, d.num_seqs + u % mix.num_prefills,
                                u / mix.num_prefills, lds);
  else
    decode_rows<Tag, CTag, WHOLE, HD, DEC_WAVES>(d, kvh, u % d.num_seqs,
                                                 u / d.num_seqs, lds);
}

}  // namespace

// Rows 0 .. num_decodes - 1 as paged_decode_attention, the others as
// prefill_attention; both in num_decodes and num_reqs at least one.
void mixed_attention(torch::Tensor out, torch::Tensor q,
                     torch::Tensor kv_cache, torch::Tensor block_table,
                     torch::Tensor query_start_loc, torch::Tensor seq_lens,
                     double scale, int64_t num_decodes,
                     int64_t max_decode_len, int64_t max_query_len,
                     int64_t sliding_window, torch::Tensor tmp_out,
                     torch::Tensor tmp_lse) {
  const int num_seqs = (int)num_decodes;
  const int num_prefills = (int)seq_lens.size(0) - num_seqs;
  const int head_dim = q.size(2);
  TORCH_CHECK(num_seqs > 0 && num_prefills > 0 && q.size(0) >= num_seqs &&
              (head_dim == 64 || head_dim == 128),
              "mixed_attention: decode rows and portions, heads of 64 or 128");
  check_prefill(out, q, kv_cache);
  const DecodePlan plan =
      plan_decode(out, q, kv_cache, num_seqs, scale, max_decode_len,
                  sliding_window, tmp_out, tmp_lse);
  const int num_kv_heads = kv_cache.size(2);
  const int tiles =
      prefill_tiles(max_query_len, (int)q.size(1) / num_kv_heads) *
      num_prefills;
  const int rows = num_seqs * plan.num_parts;
  const Mix mix{tiles, rows, std::min(tiles + rows, tiles + (tiles + 1) / 2),
                num_prefills};
  TORCH_CHECK(mix.tiles + mix.rows < 65536, "mixed_attention: grid");
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto launch = [&](auto tag, auto ctag, auto dim, auto whole) {
    using CTag = decltype(ctag);
    hipLaunchKernelGGL(
        (mixed_attention_kernel<decltype(tag), CTag, decltype(whole)::value,
                                decltype(dim)::value>),
        dim3(num_kv_heads, mix.tiles + mix.rows), dim3(PF_BLOCK), 0, stream,
        decode_args<CTag>(plan, out, q, kv_cache, num_seqs, block_table,
                          seq_lens, sliding_window, tmp_out, tmp_lse),
        prefill_args<CTag>(out, q, kv_cache, block_table, query_start_loc,
                           seq_lens, scale, sliding_window),
        mix);
  };
  const bool fp8c = kv_cache.scalar_type() == torch::kFloat8_e4m3fn;
  auto by_parts = [&](auto tag, auto ctag, auto dim) {
    if (plan.num_parts == 1) launch(tag, ctag, dim, std::true_type{});
    else                     launch(tag, ctag, dim, std::false_type{});
  };
  auto by_type = [&](auto dim) {
    if (q.scalar_type() == torch::kBFloat16) {
      if (fp8c) by_parts(BF16Tag{}, FP8CacheTag{}, dim);
      else      by_parts(BF16Tag{}, BF16Tag{}, dim);
    } else {
      if (fp8c) by_parts(FP16Tag{}, FP8CacheTag{}, dim);
      else      by_parts(FP16Tag{}, FP16Tag{}, dim);
    }
  };
  if (head_dim == 64) by_type(std::integral_constant<int, 64>{});
  else by_type(std::integral_constant<int, 128>{});
  HIP_CHECK_KERNEL();
}

}  // namespace vllm_amd
