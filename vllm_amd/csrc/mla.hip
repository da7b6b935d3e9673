// MLA attention for CDNA4 (gfx950): decode rows and prompt portions over
// the compressed latent KV cache.
//
// Absorbed-MQA form (blueprint: reference
// vllm/model_executor/layers/attention/mla_attention.py:40-190): queries
// are carried through W_UK first, so all heads of a token attend with dim
// L+R (512 + 64) against ONE shared latent stream whose first 512 dims
// are the value as well. Every cached row meets 2 * 1088 flops per head:
// with 128 heads that is 240 flops per byte, so the matrix cores bound it
// and the tile is laid out for them:
//   - A workgroup is one token and 128 heads, eight waves of 16 heads. A
//     wave keeps its queries (72 registers) and all 512 output columns
//     (128 registers) for the whole pass; two waves per SIMD fit, so one
//     wave's softmax and LDS latency run under another's products.
//     (32-head waves would read half the LDS bytes per flop, but need 400
//     registers before the first temporary.)
//   - 16x16x32 MFMA: S^T = K Q^T with the heads as columns, so a lane
//     holds 16 of 64 keys of one head and P^T is already the fragment
//     O^T = V^T P^T needs when the keys are taken in the order the score
//     registers hold them: P never leaves its lane.
//   - One LDS copy of 64 latent rows serves both products: K fragments
//     are plain 16 B reads, V^T fragments transposing reads of the same
//     rows. 16 B chunks of a row are exchanged so that neither kind of
//     read meets a bank twice.
//   - Reads run four and more products ahead of their use, in an order the
//     scheduler is told: left alone it waits for each read just before its
//     product (115 -> 90 us for the decode rows below, 1.60 -> 1.32 ms for
//     the prompts).
//   - Two such tiles alternate; they are filled straight from global
//     memory (no registers), one tile ahead, one barrier per tile.
//   - Where the weights keep more than 16 bits (hi + lo, prompts),
//     accumulators are rescaled only when a head's maximum has grown by
//     2^8. Where they are rounded to 16 (decode), the largest is kept at
//     one and the rounded weights are summed: 3 % slower, 4 % closer to
//     64-bit results.
// Rows are split over a few partitions of the keys, and heads over workgroups
// (group_heads below), when there are fewer than CUs; fp32 partials (256 KB per
// row and partition) are merged by mla_reduce_kernel, so partitions are few and
// long, and rows that fit one are written at once. A portion of 2 tokens after
// 8190 takes 56 us in 64 partitions, with the products around it, and 510 in
// one. 128 heads: 128 rows x 129..2176 keys 1025 -> 88 us with the merge (four
// waves of 16 heads on 32-key tiles, V stored transposed, before); prompts of
// 300, 1300 and 2301 tokens 1.32 ms (750 TFLOP/s counting P once; a composition
// of library products in fp32 before, 24 ms).

#include <torch/all.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include "common.h"

namespace vllm_amd {

namespace mla {

constexpr int LORA = 512;
constexpr int ROPE = 64;
constexpr int DK = LORA + ROPE;   // 576
constexpr int HG = 128;           // heads per workgroup, at most
constexpr int SUB = 64;           // keys per LDS tile
constexpr int WAVES = 8;
constexpr int THREADS = WAVES * WAVE_SIZE;
constexpr int CHUNKS = DK / 8;    // 16 B chunks per row
constexpr int TILE_BYTES = SUB * DK * 2;
constexpr int BUFS = 2;
constexpr int FILL = SUB * CHUNKS / THREADS;  // 16 B loads a thread and tile
constexpr float NEG = -3.0e38f;
constexpr float GROWTH = 8.f;

// A row is 4.5 x 256 B, so odd rows start half a bank period later. The
// eight chunks of each 128 B are exchanged by a number that differs in more
// than its last bit over rows 0..7 and 8..15 (V reads: 8 rows, two
// neighbouring chunks) and keeps a part of a K read off its own banks: 16 B
// reads are served 16 lanes at a time, lanes 0..3, 12..15, 20..23 and
// 24..27 first, that is one chunk of rows 0..3 and 12..15 and its
// neighbour of rows 4..11. (With lanes 0..15 in mind alone every K read met
// each bank twice.)
DEVINL int chunk_slot(int row, int c) {
  const int x = (row >> 1) & 7;
  return c ^ ((((x & 3) ^ ((x >> 2) << 1)) << 1) | (x >> 2));
}

// The request of a prompt token: the last one starting at or before its
// row. Returns how many keys the token sees.
DEVINL int prompt_keys(int row, const int* __restrict__ query_start_loc,
                       const int* __restrict__ seq_lens, int num_decodes,
                       int num_reqs, int& req) {
  req = num_decodes;
  for (int end = num_reqs; end - req > 1;) {
    const int mid = (req + end) / 2;
    if (query_start_loc[mid] <= row) req = mid;
    else end = mid;
  }
  return seq_lens[req] - (query_start_loc[req + 1] - 1 - row);
}

// One workgroup: (token row, partition of part_len keys, head group); the
// last partition takes what is left.
// PROMPT: blockIdx.x counts the batch's prompt tokens from the last one
// (the last tokens of a portion have most keys); otherwise blockIdx.x is a
// decode row. PARTS: blockIdx.y is a partition. SPLIT_P keeps the weights
// at more than 16 bits (hi + lo parts, two products).
template <typename Tag, bool PROMPT, bool SPLIT_P, bool PARTS>
__launch_bounds__(THREADS, 2) __global__
void mla_kernel(short* __restrict__ out,           // [T, Hq, LORA]
                const short* __restrict__ q_nope,  // [T, Hq, LORA]
                const short* __restrict__ q_pe,    // [T, Hq, ROPE]
                const short* __restrict__ kv,      // [NB, BS, DK]
                const int* __restrict__ block_table, int bt_stride,
                const int* __restrict__ query_start_loc,
                const int* __restrict__ seq_lens, float scale_log2,
                int num_heads, int block_size, int num_decodes,
                int num_reqs,
                float* __restrict__ tmp_out,  // [rows, Hq, parts, LORA]
                float* __restrict__ tmp_lse,  // [rows, Hq, parts, 2]
                int num_parts, int part_len, int group_heads) {
  int req, row, ctx, first = 0;   // first: row 0 of the scratch
  if constexpr (PROMPT) {
    row = query_start_loc[num_reqs] - 1 - (int)blockIdx.x;
    first = query_start_loc[num_decodes];
    if (row < first) return;
    ctx = prompt_keys(row, query_start_loc, seq_lens, num_decodes, num_reqs,
                      req);
  } else {
    req = row = blockIdx.x;
    ctx = seq_lens[req];
  }
  const int hg0 = blockIdx.z * group_heads;
  const int part = PARTS ? blockIdx.y : 0;
  const int t_begin = PARTS ? part * part_len : 0;
  const int t_end =
      PARTS && part + 1 < num_parts ? min(ctx, t_begin + part_len) : ctx;
  if (t_begin >= t_end) {
    if (!PROMPT && part == 0) {   // a row without keys (padding) is zero
      const int n = min(group_heads, num_heads - hg0) * (LORA / 8);
      short* ob = out + ((int64_t)row * num_heads + hg0) * LORA;
      for (int c = threadIdx.x; c < n; c += THREADS)
        *reinterpret_cast<i32x4*>(ob + c * 8) = i32x4{0, 0, 0, 0};
    }
    return;
  }

  __shared__ __align__(16) char lds[BUFS * TILE_BYTES];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  const int head = hg0 + wave * 16 + l16;
  const bool busy =
      wave * 16 < group_heads && hg0 + wave * 16 < num_heads;

  s16x8 qf[DK / 32];
  {
    const int64_t h = (int64_t)row * num_heads + min(head, num_heads - 1);
    const short* qn = q_nope + h * LORA + l4 * 8;
    const short* qp = q_pe + h * ROPE + l4 * 8;
#pragma unroll
    for (int kk = 0; kk < LORA / 32; ++kk)
      qf[kk] = *reinterpret_cast<const s16x8*>(qn + kk * 32);
#pragma unroll
    for (int kk = 0; kk < ROPE / 32; ++kk)
      qf[LORA / 32 + kk] = *reinterpret_cast<const s16x8*>(qp + kk * 32);
  }

  const int* bt = block_table + (int64_t)req * bt_stride;
  // Each wave fills 8 rows. Rows past the end repeat the last one: their
  // weight is zero, and what a stale row holds could be NaN.
  auto fill = [&](int sub0, int buf) {
    int ln = lane;
    asm("" : "+v"(ln));  // recompute the places each time: no registers
    const int last = t_end - 1 - sub0;
    char* dst = lds + buf * TILE_BYTES + wave * (FILL * WAVE_SIZE * 16);
    auto place = [&](int i, int& rr, int& e) {
      const int c = i * WAVE_SIZE + ln;
      const int r8 = c / CHUNKS;
      const int r = wave * (SUB / WAVES) + r8;
      e = chunk_slot(r, c - r8 * CHUNKS) * 8;
      rr = min(r, last);
    };
    int rr, e;
    if (block_size % SUB == 0) {   // the tile is part of one cache block
      const int b = sub0 / block_size;
      const short* base =
          kv + ((int64_t)bt[b] * block_size + (sub0 - b * block_size)) * DK;
#pragma unroll
      for (int i = 0; i < FILL; ++i) {
        place(i, rr, e);
        lds_fill16(base + (rr * DK + e), dst + i * WAVE_SIZE * 16);
      }
    } else {
      for (int i = 0; i < FILL; ++i) {
        place(i, rr, e);
        const int t = sub0 + rr;
        const int b = t / block_size;
        lds_fill16(kv + ((int64_t)bt[b] * block_size + (t - b * block_size)) *
                            DK + e,
                   dst + i * WAVE_SIZE * 16);
      }
    }
  };

  // Byte places of this lane's fragments in a tile. The exchange of chunks
  // only touches the low three bits of a chunk and repeats every 16 rows,
  // so all other parts of an address are constants.
  int k_at[2], v_at[4];
  k_at[0] = l16 * (DK * 2) + chunk_slot(l16, l4) * 16;
  k_at[1] = k_at[0] ^ 64;
  {
    const int r = l4 * 4 + (l16 >> 2);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v_at[j] = r * (DK * 2) + chunk_slot(r, j * 2 + ((l16 & 3) >> 1)) * 16 +
                (l16 & 1) * 8;
  }

  float m_run = NEG, l_run = 0.f;  // of this head, log2 domain; l: own keys
  f32x4 o[LORA / 16];
#pragma unroll
  for (int i = 0; i < LORA / 16; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  fill(t_begin, 0);
  int buf = 0;
  for (int sub0 = t_begin; sub0 < t_end; sub0 += SUB, buf ^= 1) {
    // The tile has landed for this wave, then for all; and every wave is
    // done with the tile before, whose place the next one takes.
    lds_fill_wait();
    __syncthreads();
    if (sub0 + SUB < t_end) fill(sub0 + SUB, buf ^ 1);
    if (!busy) continue;
    const char* t = lds + buf * TILE_BYTES;
    // ---- S^T: 64 keys x 16 heads -----------------------------------------
    f32x4 s[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) s[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < DK / 32; ++kk)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const s16x8 a = *reinterpret_cast<const s16x8*>(
            t + k_at[kk & 1] + n * 16 * (DK * 2) + (kk >> 1) * 128);
        s[n] = mfma16<Tag>(a, qf[kk], s[n]);
      }
    reads_ahead<4, 1, DK / 32 * 4>();
    // ---- softmax: s[n][r] is key n*16 + l4*4 + r -------------------------
    const int left = t_end - sub0 - l4 * 4;
    float mx = NEG;
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[n][r] = n * 16 + r < left ? s[n][r] * scale_log2 : NEG;
        mx = __builtin_amdgcn_fmed3f(mx, s[n][r], INFINITY);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx - m_run > (SPLIT_P ? GROWTH : 0.f))) {
      const float m_new = fmaxf(m_run, mx);
      const float f = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= f;
#pragma unroll
      for (int i = 0; i < LORA / 16; ++i) o[i] *= f;
      m_run = m_new;
    }
    // ---- O^T += V^T P^T, 32 keys at a time -------------------------------
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      i32x4 hi, lo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4& sc = s[c * 2 + (j >> 1)];
        const float p0 = __builtin_amdgcn_exp2f(sc[(j & 1) * 2] - m_run);
        const float p1 = __builtin_amdgcn_exp2f(sc[(j & 1) * 2 + 1] - m_run);
        hi[j] = pack2<Tag>(p0, p1);
        l_run = SPLIT_P ? l_run + (p0 + p1) : add_pair<Tag>(hi[j], l_run);
        lo[j] = SPLIT_P ? pack2<Tag>(p0 - unpack_lo<Tag>(hi[j]),
                                     p1 - unpack_hi<Tag>(hi[j])) : 0;
      }
      const s16x8 p_hi = __builtin_bit_cast(s16x8, hi);
      const s16x8 p_lo = __builtin_bit_cast(s16x8, lo);
#pragma unroll
      for (int i = 0; i < LORA / 16; ++i) {
        const char* at = t + v_at[i & 3] + c * 32 * (DK * 2) + (i >> 2) * 128;
        const s16x4 a = lds_read_tr(at);
        const s16x4 b = lds_read_tr(at + 16 * (DK * 2));
        const s16x8 v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
        if constexpr (SPLIT_P) o[i] = mfma16<Tag>(v, p_lo, o[i]);
        o[i] = mfma16<Tag>(v, p_hi, o[i]);
      }
      reads_ahead<SPLIT_P ? 4 : 8, 2, LORA / 16, SPLIT_P ? 2 : 1>();
    }
  }

  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (!busy || head >= num_heads) return;
  const int64_t hrow = (int64_t)row * num_heads + head;
  if (!PARTS || num_parts == 1 || ctx <= part_len) {   // nothing to merge
    const float inv_l = 1.f / l_run;
    short* ob = out + hrow * LORA + l4 * 4;
#pragma unroll
    for (int i = 0; i < LORA / 16; ++i) {
      int2 v;
      v.x = pack2<Tag>(o[i][0] * inv_l, o[i][1] * inv_l);
      v.y = pack2<Tag>(o[i][2] * inv_l, o[i][3] * inv_l);
      *reinterpret_cast<int2*>(ob + i * 16) = v;
    }
  } else {
    const int64_t at =
        ((int64_t)(row - first) * num_heads + head) * num_parts + part;
    float* ob = tmp_out + at * LORA + l4 * 4;
#pragma unroll
    for (int i = 0; i < LORA / 16; ++i)
      *reinterpret_cast<f32x4*>(ob + i * 16) = o[i];
    if (l4 == 0) {
      tmp_lse[at * 2] = m_run;
      tmp_lse[at * 2 + 1] = l_run;
    }
  }
}

// Merge partitions: out[s,h,:] = sum_p w_p * tmp[s,h,p,:] / sum_p w_p l_p
// with w_p = exp2(m_p - m_max). One wave per (row, head), 8 columns each.
template <typename Tag, bool PROMPT>
__launch_bounds__(WAVE_SIZE) __global__
void mla_reduce_kernel(short* __restrict__ out,
                       const float* __restrict__ tmp_out,
                       const float* __restrict__ tmp_lse,
                       const int* __restrict__ query_start_loc,
                       const int* __restrict__ seq_lens, int num_decodes,
                       int num_reqs, int num_heads, int num_parts,
                       int part_len) {
  const int h = blockIdx.x;
  int row = blockIdx.y, ctx;
  const int64_t trow = (int64_t)row * num_heads + h;
  if constexpr (PROMPT) {
    int req;
    row += query_start_loc[num_decodes];
    if (row >= query_start_loc[num_reqs]) return;
    ctx = prompt_keys(row, query_start_loc, seq_lens, num_decodes, num_reqs,
                      req);
  } else {
    ctx = seq_lens[row];
  }
  const int parts = min((ctx + part_len - 1) / part_len, num_parts);
  if (parts <= 1) return;   // the row fits one partition: it is done
  const int64_t hrow = (int64_t)row * num_heads + h;
  const float* lse = tmp_lse + trow * num_parts * 2;
  float m = NEG;
  for (int p = 0; p < parts; ++p) m = fmaxf(m, lse[p * 2]);
  float l = 0.f;
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  const float* src = tmp_out + trow * num_parts * LORA + threadIdx.x * 8;
#pragma unroll 4
  for (int p = 0; p < parts; ++p) {
    const float w = __builtin_amdgcn_exp2f(lse[p * 2] - m);
    l += w * lse[p * 2 + 1];
    acc[0] += w * *reinterpret_cast<const f32x4*>(src + (int64_t)p * LORA);
    acc[1] += w * *reinterpret_cast<const f32x4*>(src + (int64_t)p * LORA + 4);
  }
  const float inv_l = 1.f / l;
  i32x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    v[j] = pack2<Tag>(acc[j >> 1][(j & 1) * 2] * inv_l,
                      acc[j >> 1][(j & 1) * 2 + 1] * inv_l);
  *reinterpret_cast<i32x4*>(out + hrow * LORA + threadIdx.x * 8) = v;
}

static void check(const torch::Tensor& out, const torch::Tensor& q_nope,
                  const torch::Tensor& q_pe, const torch::Tensor& kv_cache) {
  TORCH_CHECK(q_nope.dim() == 3 && q_nope.size(2) == LORA,
              "mla kernel expects kv_lora_rank=512");
  TORCH_CHECK(q_pe.size(2) == ROPE, "mla kernel expects rope dim 64");
  TORCH_CHECK(kv_cache.size(2) == DK);
  TORCH_CHECK(q_nope.is_contiguous() && q_pe.is_contiguous() &&
              out.is_contiguous() && kv_cache.is_contiguous() &&
              (uintptr_t)kv_cache.data_ptr() % 16 == 0);
  TORCH_CHECK(out.scalar_type() == q_nope.scalar_type() &&
              q_pe.scalar_type() == q_nope.scalar_type() &&
              kv_cache.scalar_type() == q_nope.scalar_type());
  TORCH_CHECK(q_nope.scalar_type() == torch::kBFloat16 ||
                  q_nope.scalar_type() == torch::kHalf,
              "mla kernel: bf16/fp16 only");
}

// Into how many partitions scratch [rows, Hq, parts, 512] and
// [rows, Hq, parts, 2] splits the keys; empty means one.
static int parts_of(const torch::Tensor& tmp_out,
                    const torch::Tensor& tmp_lse, int64_t rows, int64_t Hq) {
  if (tmp_out.numel() == 0) return 1;
  TORCH_CHECK(tmp_out.dim() == 4 && tmp_lse.dim() == 4 &&
              tmp_out.is_contiguous() && tmp_lse.is_contiguous() &&
              tmp_out.size(0) == rows && tmp_lse.size(0) == rows &&
              tmp_out.size(1) == Hq && tmp_lse.size(1) == Hq &&
              tmp_out.size(2) == tmp_lse.size(2) &&
              tmp_out.size(3) == LORA && tmp_lse.size(3) == 2,
              "mla scratch must be [rows, Hq, parts, 512] and "
              "[rows, Hq, parts, 2]");
  return (int)tmp_out.size(2);
}

static int part_length(int64_t max_seq_len, int parts) {
  return ceil_div(ceil_div((int)std::max<int64_t>(max_seq_len, 1), parts),
                  SUB) * SUB;
}

// Heads that a workgroup takes, of `pairs` rows and partitions: fewer than 128
// while a round of workgroups then still has room on 256 CUs. A tile of 64
// heads takes two thirds of the time of one of 128, of 32 half, and each
// workgroup reads its queries and writes its partials in proportion, so few
// and short rows are done sooner, and others need fewer partitions. us at 128
// heads with the merge, 128 / 64 / 32 heads a workgroup, each in its best
// number of partitions: 1 x 200 keys 21.6 / 14.2 / 12.3, 1 x 4000 28.8 / 24.2 /
// 22.0, 8 x 4000 37.0 / 31.4 / 34.7, 64 x 100..150 27.4 / 17.9 / 16.1, 76 x
// 431..531 40.9 / 33.6, 128 x 1000 64.8 / 57.7; 32 x 8192 103 / 106, 128 x
// 129..2176 85 / 96 (hip_ops.py chooses the partitions with this in mind).
static int group_heads(int64_t pairs, int64_t Hq) {
  int n = HG;
  while (n > 32 && Hq > n / 2 && pairs * ceil_div((int)Hq, n / 2) <= 256)
    n /= 2;
  return n;
}

}  // namespace mla

int64_t mla_group_heads(int64_t pairs, int64_t heads) {
  return mla::group_heads(pairs, heads);
}

// Decode rows; the scratch says into how many partitions their keys go.
void mla_decode(torch::Tensor out, torch::Tensor q_nope, torch::Tensor q_pe,
                torch::Tensor kv_cache, torch::Tensor block_table,
                torch::Tensor seq_lens, double scale, int64_t max_seq_len,
                torch::Tensor tmp_out, torch::Tensor tmp_lse) {
  using namespace mla;
  check(out, q_nope, q_pe, kv_cache);
  const int T = (int)q_nope.size(0);
  if (T == 0) return;
  const int Hq = (int)q_nope.size(1);
  const int bs = (int)kv_cache.size(1);
  const int parts = parts_of(tmp_out, tmp_lse, T, Hq);
  const int part_len = part_length(max_seq_len, parts);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const int heads = group_heads((int64_t)T * parts, Hq);
  dim3 grid(T, parts, ceil_div(Hq, heads));
  auto launch = [&](auto tag) {
    using Tag = decltype(tag);
    hipLaunchKernelGGL(
        (mla_kernel<Tag, false, false, true>), grid, dim3(THREADS), 0, stream,
        (short*)out.data_ptr(), (const short*)q_nope.data_ptr(),
        (const short*)q_pe.data_ptr(), (const short*)kv_cache.data_ptr(),
        block_table.data_ptr<int>(), (int)block_table.size(1), nullptr,
        seq_lens.data_ptr<int>(), (float)scale * 1.4426950408889634f, Hq, bs,
        T, T, parts > 1 ? tmp_out.data_ptr<float>() : nullptr,
        parts > 1 ? tmp_lse.data_ptr<float>() : nullptr, parts, part_len,
        heads);
    if (parts > 1) {
      HIP_CHECK_KERNEL();
      hipLaunchKernelGGL((mla_reduce_kernel<Tag, false>), dim3(Hq, T),
                         dim3(WAVE_SIZE), 0, stream, (short*)out.data_ptr(),
                         tmp_out.data_ptr<float>(), tmp_lse.data_ptr<float>(),
                         nullptr, seq_lens.data_ptr<int>(), T, T, Hq, parts,
                         part_len);
    }
  };
  if (q_nope.scalar_type() == torch::kBFloat16) launch(BF16Tag{});
  else launch(FP16Tag{});
  HIP_CHECK_KERNEL();
}

// Prompt portions: requests num_decodes.. of the batch; q/out cover the
// whole step, the scratch the prompt tokens.
void mla_prefill(torch::Tensor out, torch::Tensor q_nope, torch::Tensor q_pe,
                 torch::Tensor kv_cache, torch::Tensor block_table,
                 torch::Tensor query_start_loc, torch::Tensor seq_lens,
                 double scale, int64_t num_decodes, int64_t max_seq_len,
                 torch::Tensor tmp_out, torch::Tensor tmp_lse) {
  using namespace mla;
  check(out, q_nope, q_pe, kv_cache);
  const int reqs = (int)seq_lens.size(0);
  const int rows = (int)(q_nope.size(0) - num_decodes);
  if (reqs <= num_decodes || rows <= 0) return;
  TORCH_CHECK(query_start_loc.numel() > reqs);
  const int Hq = (int)q_nope.size(1);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const int parts = parts_of(tmp_out, tmp_lse, rows, Hq);
  const int part_len = part_length(max_seq_len, parts);
  const int heads = group_heads((int64_t)rows * parts, Hq);
  dim3 grid(rows, parts, ceil_div(Hq, heads));
  auto launch = [&](auto tag, auto split) {
    using Tag = decltype(tag);
    constexpr bool PARTS = decltype(split)::value;
    hipLaunchKernelGGL(
        (mla_kernel<Tag, true, true, PARTS>), grid, dim3(THREADS), 0, stream,
        (short*)out.data_ptr(), (const short*)q_nope.data_ptr(),
        (const short*)q_pe.data_ptr(), (const short*)kv_cache.data_ptr(),
        block_table.data_ptr<int>(), (int)block_table.size(1),
        query_start_loc.data_ptr<int>(), seq_lens.data_ptr<int>(),
        (float)scale * 1.4426950408889634f, Hq, (int)kv_cache.size(1),
        (int)num_decodes, reqs, PARTS ? tmp_out.data_ptr<float>() : nullptr,
        PARTS ? tmp_lse.data_ptr<float>() : nullptr, parts, part_len,
        heads);
    if constexpr (PARTS) {
      HIP_CHECK_KERNEL();
      hipLaunchKernelGGL((mla_reduce_kernel<Tag, true>), dim3(Hq, rows),
                         dim3(WAVE_SIZE), 0, stream, (short*)out.data_ptr(),
                         tmp_out.data_ptr<float>(), tmp_lse.data_ptr<float>(),
                         query_start_loc.data_ptr<int>(),
                         seq_lens.data_ptr<int>(), (int)num_decodes, reqs, Hq,
                         parts, part_len);
    }
  };
  auto by_parts = [&](auto tag) {
    if (parts > 1) launch(tag, std::true_type{});
    else           launch(tag, std::false_type{});
  };
  if (q_nope.scalar_type() == torch::kBFloat16) by_parts(BF16Tag{});
  else by_parts(FP16Tag{});
  HIP_CHECK_KERNEL();
}

}  // namespace vllm_amd
