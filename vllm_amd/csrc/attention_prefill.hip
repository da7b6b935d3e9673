// Flash-style varlen prefill attention over the paged KV cache for
// MI355X (gfx950, CDNA4).
//
// What bounds it: the matrix cores, with the exponentials and LDS reads
// close behind (per 32 x 64 scores of a wave: 1024 cycles of MFMA at
// D=128, about as many of vector ALU and, over four waves, of LDS). So:
//   - 32x32x16 MFMA, four waves of 32 rows: half the LDS bytes per flop
//     of 16-row fragments. Two workgroups per CU fit at D=128, so one
//     wave's softmax runs under another's products.
//   - The rows of a tile are (token, query head) pairs of ONE KV head:
//     the heads of a group share every K/V tile they read, the causal
//     edge of a tile is only 128 / group tokens wide, and a short
//     portion still fills its tile.
//   - Scores are S^T = K Q^T: a lane holds 32 keys of one row, so the
//     row maximum is 31 in-lane steps and one half-wave swap, maximum
//     and sum stay in registers, and the 16-bit P^T is already the
//     fragment that O^T = V^T P^T needs when the contraction runs over
//     the keys in the order in which the score registers hold them.
//   - V^T fragments come from transposing LDS reads of the row-major
//     tile: no scatter when the tile is stored.
//   - K/V tiles are double-buffered: the tile after next is in flight in
//     registers while two are in LDS, one barrier per tile.
//   - The 16-bit weights are summed as they are rounded (one dot product
//     instruction a pair), so that their rounding cancels in the quotient,
//     and the row's largest weight is exactly one: accumulators are
//     rescaled whenever a maximum moves. Letting it grow by 2^8 first
//     would save 3 % and raise the distance to 64-bit results by 2 to 7 %
//     (now 1 % below that of unrounded sums).
//   - Results are stored 16 B a lane (8 B: 59 us for the short prompts
//     below, 53 now).
// Against 16x16x32 fragments on 16-row waves with V scattered into LDS:
// one 8192-token prompt, 32/8 heads of 128: 4.70 -> 0.67 ms (820 TFLOP/s);
// 64 prompts of 33..223 tokens: 207 -> 54 us; 4 x 2048 tokens, 16/8 heads
// of 256: 2.59 -> 0.26 ms.
//
// Role of the reference's triton_unified_attention.py:179 (prefill side)
// and prefix_prefill.py.

#include <torch/all.h>
#include <c10/hip/HIPStream.h>

#include "common.h"

namespace vllm_amd {

constexpr int PF_WAVES = 4;
constexpr int PF_BLOCK = PF_WAVES * WAVE_SIZE;
constexpr int PF_ROWS = PF_WAVES * 32;  // (token, head) rows per workgroup
constexpr int KVTILE = 64;     // keys per inner tile == cache block_size
constexpr float LOG2E = 1.4426950408889634f;
constexpr float PF_NEG = -3.0e38f;

// 16 B chunk of a K row: the 16 rows that one phase of a fragment read
// takes the same chunk from land on different banks (64 x 4 B).
template <int HD> DEVINL int k_chunk(int row, int c) {
  if constexpr (HD == 64) return c ^ ((row >> 1) & 7);
  return c ^ (row & 15);
}
// 32 B segment of a V row: a transposing read takes two neighbouring
// segments of four consecutive rows per half wave.
template <int HD> DEVINL int v_seg(int row, int s) {
  if constexpr (HD == 64) return s ^ (((row >> 1) & 1) << 1);
  return s ^ ((row & 3) << 1);
}

// Maximum over a lane and its counterpart in the other half wave.
DEVINL float half_max(float x) {
  const auto sw = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  const unsigned lo = sw[0], hi = sw[1];
  return fmaxf(__uint_as_float(lo), __uint_as_float(hi));
}

template <typename Tag, typename CTag, int HD>
__global__ __launch_bounds__(PF_BLOCK, HD == 256 ? 1 : 2)
void prefill_attention_kernel(
    short* __restrict__ out,             // [T, Hq, D]
    const short* __restrict__ q,         // [T, Hq, D]
    const typename CacheTraits<CTag>::elem* __restrict__ kv_cache,
                                         // [2, blocks, Hkv, 64, D]
    const int* __restrict__ block_table, // [num_reqs, max_blocks]
    const int* __restrict__ query_start_loc,  // [num_reqs+1]
    const int* __restrict__ seq_lens,         // [num_reqs]
    const float scale_log2, const int negate, const int group,
    const int num_kv_heads, const int max_blocks_per_req,
    const int num_decodes, const int64_t kv_plane_stride,
    const int64_t q_stride, const int sliding_window) {
  using elem = typename CacheTraits<CTag>::elem;
  constexpr bool FP8 = sizeof(elem) == 1;
  constexpr int EPV = 16 / sizeof(elem);              // elements per 16 B
  constexpr int LD = KVTILE * HD / EPV / PF_BLOCK;    // 16 B loads a thread
  constexpr int KF = HD / 16;                         // MFMA steps over D
  constexpr int DS = HD / 32;                         // output row tiles
  constexpr int TILE = KVTILE * HD;                   // 16-bit elements

  // One XCD takes every eighth workgroup, so with the KV head fastest a
  // head's tiles stay in one L2. Late tiles attend most keys: first.
  const int kvh = blockIdx.x;
  const int req = num_decodes + blockIdx.z;
  const int q_start = query_start_loc[req];
  const int ql = query_start_loc[req + 1] - q_start;
  const int rows = ql * group;
  const int tile = (rows + PF_ROWS - 1) / PF_ROWS - 1 - (int)blockIdx.y;
  if (tile < 0) return;
  const int row0 = tile * PF_ROWS;
  const int ctx = seq_lens[req];
  const int num_q_heads = num_kv_heads * group;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l32 = lane & 31;
  const int half = lane >> 5;

  __shared__ __align__(16) short k_lds[2][TILE];   // [tok][d], chunks moved
  __shared__ __align__(16) short v_lds[2][TILE];   // [tok][d], segments moved

  // --- this lane's row: token and head --------------------------------
  const int row = row0 + wave * 32 + l32;
  const int row_safe = min(row, rows - 1);
  const int tok = row_safe / group;
  const int head = kvh * group + row_safe % group;
  const int pos0 = ctx - ql;          // position of the first new token
  const int qpos = pos0 + tok;

  s16x8 qf[KF];
  {
    const short* qb = q + (int64_t)(q_start + tok) * q_stride +
                      (int64_t)head * HD + half * 8;
#pragma unroll
    for (int kk = 0; kk < KF; ++kk) {
      i32x4 v = *reinterpret_cast<const i32x4*>(qb + kk * 16);
      if (negate) v ^= i32x4{(int)0x80008000, (int)0x80008000,
                             (int)0x80008000, (int)0x80008000};
      qf[kk] = __builtin_bit_cast(s16x8, v);
    }
  }

  float m_run = PF_NEG, l_run = 0.f;  // maximum (unscaled) of the row; sum
                                      // over the keys this lane holds
  f32x16 o[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;

  // Keys the tile's first and last rows see.
  const int first_pos = pos0 + row0 / group;
  const int last_pos = pos0 + (min(row0 + PF_ROWS, rows) - 1) / group;
  const int kt0 =
      sliding_window > 0 ? max(0, first_pos - sliding_window + 1) / KVTILE : 0;
  const int kt_end = last_pos / KVTILE + 1;

  const int* bt = block_table + (int64_t)req * max_blocks_per_req;
  i32x4 kr[LD], vr[LD];
  auto load = [&](int phys) {
    const elem* src =
        kv_cache + ((int64_t)phys * num_kv_heads + kvh) * (KVTILE * HD);
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      kr[i] = *reinterpret_cast<const i32x4*>(
          src + (i * PF_BLOCK + threadIdx.x) * EPV);
      vr[i] = *reinterpret_cast<const i32x4*>(
          src + kv_plane_stride + (i * PF_BLOCK + threadIdx.x) * EPV);
    }
  };
  auto store = [&](int kt) {
    const int b = kt & 1;
    if (kt * KVTILE + KVTILE > ctx) {
      // Rows no token has been written to yet may hold anything, and
      // their zero weight does not stop a NaN.
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const int key = kt * KVTILE + (i * PF_BLOCK + threadIdx.x) * EPV / HD;
#pragma unroll
        for (int j = 0; j < 4; ++j) vr[i][j] = key < ctx ? vr[i][j] : 0;
      }
    }
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int e = (i * PF_BLOCK + threadIdx.x) * EPV;
      const int r = e / HD;
      const int c = (e % HD) / 8;
#pragma unroll
      for (int h = 0; h < EPV / 8; ++h) {
        i32x4 kv, vv;
        if constexpr (FP8) {
          const int2 a = fp8x4_widen<Tag>(kr[i][h * 2]);
          const int2 bb = fp8x4_widen<Tag>(kr[i][h * 2 + 1]);
          kv = i32x4{a.x, a.y, bb.x, bb.y};
          const int2 x = fp8x4_widen<Tag>(vr[i][h * 2]);
          const int2 y = fp8x4_widen<Tag>(vr[i][h * 2 + 1]);
          vv = i32x4{x.x, x.y, y.x, y.y};
        } else {
          kv = kr[i];
          vv = vr[i];
        }
        *reinterpret_cast<i32x4*>(
            &k_lds[b][r * HD + k_chunk<HD>(r, c + h) * 8]) = kv;
        *reinterpret_cast<i32x4*>(
            &v_lds[b][r * HD + v_seg<HD>(r, (c + h) >> 1) * 16 +
                      ((c + h) & 1) * 8]) = vv;
      }
    }
  };

  load(bt[kt0]);
  store(kt0);
  if (kt0 + 1 < kt_end) load(bt[kt0 + 1]);
  int phys = bt[min(kt0 + 2, kt_end - 1)];
  __syncthreads();

  for (int kt = kt0; kt < kt_end; ++kt) {
    const int b = kt & 1;
    // --- S^T: 64 keys x 32 rows -----------------------------------------
    f32x16 s[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[n][r] = 0.f;
      const int key = n * 32 + l32;
#pragma unroll
      for (int kk = 0; kk < KF; ++kk) {
        const s16x8 a = *reinterpret_cast<const s16x8*>(
            &k_lds[b][key * HD + k_chunk<HD>(key, kk * 2 + half) * 8]);
        s[n] = mfma32<Tag>(a, qf[kk], s[n]);
      }
    }
    // The other buffer was last read before the barrier that opened this
    // iteration.
    if (kt + 1 < kt_end) store(kt + 1);
    if (kt + 2 < kt_end) {
      load(phys);
      phys = bt[min(kt + 3, kt_end - 1)];
    }

    // --- mask, only where the tile meets an edge -------------------------
    // Register r of subtile n is key n*32 + 8*(r/4) + 4*half + r%4.
    const int key_base = kt * KVTILE + half * 4;
    if (kt * KVTILE + KVTILE - 1 > first_pos ||
        (sliding_window > 0 && kt * KVTILE <= last_pos - sliding_window)) {
      const int lo = sliding_window > 0 ? qpos - sliding_window : -1;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = key_base + n * 32 + 8 * (r >> 2) + (r & 3);
          s[n][r] = (key <= qpos) & (key > lo) ? s[n][r] : PF_NEG;
        }
    }

    // --- running softmax --------------------------------------------------
    // med3 with +inf is a maximum that the compiler fuses in threes (fmaxf
    // first quiets each score: 37 more instructions a tile, 2 %).
    float mx = PF_NEG;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      mx = __builtin_amdgcn_fmed3f(mx, s[0][r], INFINITY);
      mx = __builtin_amdgcn_fmed3f(mx, s[1][r], INFINITY);
    }
    mx = half_max(mx);
    if (__any(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      const float f = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2);
      l_run *= f;
#pragma unroll
      for (int i = 0; i < DS; ++i) o[i] *= f;
      m_run = m_new;
    }
    // A row that has seen no key yet (a window's first tile) weighs none.
    const float shift = m_run > PF_NEG ? -m_run * scale_log2 : 0.f;
    s16x8 pf[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      i32x4 pk;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = (c & 1) * 8 + j * 2;
        const float p0 = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[c >> 1][r], scale_log2, shift));
        const float p1 = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[c >> 1][r + 1], scale_log2, shift));
        pk[j] = pack2<Tag>(p0, p1);
        l_run = add_pair<Tag>(pk[j], l_run);
      }
      pf[c] = __builtin_bit_cast(s16x8, pk);
    }

    // --- O^T += V^T P^T ----------------------------------------------------
    const int vrow = half * 4 + ((lane & 15) >> 2);
    const int vcol = (lane & 3) * 4;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int r0 = c * 16 + vrow;
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        const int seg = i * 2 + ((lane >> 4) & 1);
        const s16x4 a = lds_read_tr(
            &v_lds[b][r0 * HD + v_seg<HD>(r0, seg) * 16 + vcol]);
        const s16x4 d = lds_read_tr(
            &v_lds[b][(r0 + 8) * HD + v_seg<HD>(r0 + 8, seg) * 16 + vcol]);
        o[i] = mfma32<Tag>(
            __builtin_shufflevector(a, d, 0, 1, 2, 3, 4, 5, 6, 7), pf[c],
            o[i]);
      }
    }
    __syncthreads();
  }

  // --- epilogue: column l32 is this lane's row ---------------------------
  l_run += __shfl_xor(l_run, 32, 64);
  const float inv_l = l_run > 0.f || l_run != l_run ? 1.f / l_run : 0.f;
  short* ob = out + ((int64_t)(q_start + tok) * num_q_heads + head) * HD +
              half * 8;
#pragma unroll
  for (int i = 0; i < DS; ++i) {
    o[i] *= inv_l;
#pragma unroll
    for (int b = 0; b < 4; b += 2) {
      const i32x4 v = row_chunk<Tag>(o[i], b);
      if (row < rows) *reinterpret_cast<i32x4*>(ob + i * 32 + b * 8) = v;
    }
  }
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
  const int group = num_q_heads / num_kv_heads;
  const int max_tiles =
      (int)((max_query_len * group + PF_ROWS - 1) / PF_ROWS);
  // The kernel takes row maxima before scaling: a negative scale moves
  // to the queries, and a scale of zero is a tiny one (all keys equal).
  const float scale_log2 =
      std::max(std::fabs((float)scale * LOG2E), 1e-30f);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  dim3 grid(num_kv_heads, max_tiles, num_prefills);

#define LAUNCH_PF(TAG, CTAG)                                                 \
  hipLaunchKernelGGL((prefill_attention_kernel<TAG, CTAG, D>), grid,         \
                     dim3(PF_BLOCK),                                         \
                     0, stream, (short*)out.data_ptr(),                      \
                     (const short*)q.data_ptr(),                             \
                     (const CacheTraits<CTAG>::elem*)kv_cache.data_ptr(),    \
                     block_table.data_ptr<int>(),                            \
                     query_start_loc.data_ptr<int>(),                        \
                     seq_lens.data_ptr<int>(), scale_log2, (int)(scale < 0), \
                     group, num_kv_heads, (int)block_table.size(1),          \
                     (int)num_decodes, kv_cache.stride(0),                   \
                     q.stride(0), (int)sliding_window)

  const bool fp8c = kv_cache.scalar_type() == torch::kFloat8_e4m3fn;
  auto dispatch = [&](auto dtag) {
    constexpr int D = decltype(dtag)::value;
    if (q.scalar_type() == torch::kBFloat16) {
      if (fp8c) { LAUNCH_PF(BF16Tag, FP8CacheTag); }
      else      { LAUNCH_PF(BF16Tag, BF16Tag); }
    } else {
      if (fp8c) { LAUNCH_PF(FP16Tag, FP8CacheTag); }
      else      { LAUNCH_PF(FP16Tag, FP16Tag); }
    }
  };
  if (head_dim == 64) dispatch(std::integral_constant<int, 64>{});
  else if (head_dim == 128) dispatch(std::integral_constant<int, 128>{});
  else dispatch(std::integral_constant<int, 256>{});
#undef LAUNCH_PF
  HIP_CHECK_KERNEL();
}

}  // namespace vllm_amd
