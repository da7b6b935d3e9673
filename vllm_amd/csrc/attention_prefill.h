// Flash-style varlen prefill attention over the paged KV cache for
// MI355X (gfx950, CDNA4): the work of a workgroup (kernels:
// attention_prefill.hip, and attention_mixed.hip beside decode rows).
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

#pragma once

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

template <typename CTag> struct PrefillArgs {
  short* out;            // [T, Hq, D]
  const short* q;        // [T, Hq, D]
  const typename CacheTraits<CTag>::elem* kv_cache;  // [2, blocks, Hkv, 64, D]
  const int* block_table;      // [num_reqs, max_blocks]
  const int* query_start_loc;  // [num_reqs+1]
  const int* seq_lens;         // [num_reqs]
  float scale_log2;
  int negate, group, num_kv_heads, max_blocks_per_req;
  int64_t kv_plane_stride, q_stride;
  int sliding_window;
};

// Bytes of LDS of a workgroup: two tiles each of keys and of values.
template <int HD> constexpr int pf_lds = 4 * KVTILE * HD * 2;

// Tile `from_last` of a request's rows, counted from the last one.
template <typename Tag, typename CTag, int HD>
DEVINL void prefill_tile(const PrefillArgs<CTag>& a, const int kvh,
                         const int req, const int from_last, char* lds) {
  using elem = typename CacheTraits<CTag>::elem;
  constexpr bool FP8 = sizeof(elem) == 1;
  constexpr int EPV = 16 / sizeof(elem);              // elements per 16 B
  constexpr int LD = KVTILE * HD / EPV / PF_BLOCK;    // 16 B loads a thread
  constexpr int KF = HD / 16;                         // MFMA steps over D
  constexpr int DS = HD / 32;                         // output row tiles
  constexpr int TILE = KVTILE * HD;                   // 16-bit elements

  const int group = a.group, num_kv_heads = a.num_kv_heads;
  const int sliding_window = a.sliding_window;
  const float scale_log2 = a.scale_log2;
  const int64_t kv_plane_stride = a.kv_plane_stride;
  const int q_start = load_uniform(a.query_start_loc + req);
  const int ql = load_uniform(a.query_start_loc + req + 1) - q_start;
  const int rows = ql * group;
  const int tile = (rows + PF_ROWS - 1) / PF_ROWS - 1 - from_last;
  if (tile < 0) return;
  const int row0 = tile * PF_ROWS;
  const int ctx = load_uniform(a.seq_lens + req);
  const int num_q_heads = num_kv_heads * group;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l32 = lane & 31;
  const int half = lane >> 5;

  // [tok][d], chunks moved; [tok][d], segments moved
  auto* k_lds = reinterpret_cast<short(*)[TILE]>(lds);
  auto* v_lds = reinterpret_cast<short(*)[TILE]>(lds + 2 * TILE * 2);

  // --- this lane's row: token and head --------------------------------
  const int row = row0 + wave * 32 + l32;
  const int row_safe = min(row, rows - 1);
  const int tok = row_safe / group;
  const int head = kvh * group + row_safe % group;
  const int pos0 = ctx - ql;          // position of the first new token
  const int qpos = pos0 + tok;

  s16x8 qf[KF];
  {
    const short* qb = a.q + (int64_t)(q_start + tok) * a.q_stride +
                      (int64_t)head * HD + half * 8;
#pragma unroll
    for (int kk = 0; kk < KF; ++kk) {
      i32x4 v = *reinterpret_cast<const i32x4*>(qb + kk * 16);
      if (a.negate) v ^= i32x4{(int)0x80008000, (int)0x80008000,
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

  const int* bt = a.block_table + (int64_t)req * a.max_blocks_per_req;
  i32x4 kr[LD], vr[LD];
  auto load = [&](int phys) {
    const elem* src =
        a.kv_cache + ((int64_t)phys * num_kv_heads + kvh) * (KVTILE * HD);
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
          const int2 k0 = fp8x4_widen<Tag>(kr[i][h * 2]);
          const int2 k1 = fp8x4_widen<Tag>(kr[i][h * 2 + 1]);
          kv = i32x4{k0.x, k0.y, k1.x, k1.y};
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

  load(load_uniform(bt + kt0));
  store(kt0);
  if (kt0 + 1 < kt_end) load(load_uniform(bt + kt0 + 1));
  int phys = load_uniform(bt + min(kt0 + 2, kt_end - 1));
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
        const s16x8 f = *reinterpret_cast<const s16x8*>(
            &k_lds[b][key * HD + k_chunk<HD>(key, kk * 2 + half) * 8]);
        s[n] = mfma32<Tag>(f, qf[kk], s[n]);
      }
    }
    // The other buffer was last read before the barrier that opened this
    // iteration.
    if (kt + 1 < kt_end) store(kt + 1);
    if (kt + 2 < kt_end) {
      load(phys);
      phys = load_uniform(bt + min(kt + 3, kt_end - 1));
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
        const s16x4 c0 = lds_read_tr(
            &v_lds[b][r0 * HD + v_seg<HD>(r0, seg) * 16 + vcol]);
        const s16x4 c1 = lds_read_tr(
            &v_lds[b][(r0 + 8) * HD + v_seg<HD>(r0 + 8, seg) * 16 + vcol]);
        o[i] = mfma32<Tag>(
            __builtin_shufflevector(c0, c1, 0, 1, 2, 3, 4, 5, 6, 7), pf[c],
            o[i]);
      }
    }
    __syncthreads();
  }

  // --- epilogue: column l32 is this lane's row ---------------------------
  l_run += __shfl_xor(l_run, 32, 64);
  const float inv_l = l_run > 0.f || l_run != l_run ? 1.f / l_run : 0.f;
  short* ob = a.out + ((int64_t)(q_start + tok) * num_q_heads + head) * HD +
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

}  // namespace vllm_amd
