// Flash-style varlen prefill attention over the paged KV cache for
// MI355X (gfx950, CDNA4): the work of a workgroup (kernels:
// attention_prefill.hip, and attention_mixed.hip beside decode rows).
//
// What bounds it: the matrix cores, with the exponentials close behind (per
// 32 x 64 scores of a wave at D=128: 1024 cycles of MFMA, about as many of
// vector ALU, half as many of LDS), and over milliseconds the chip's power
// (1.75 GHz). So:
//   - 32x32x16 MFMA, four waves of 32 rows: half the LDS bytes per flop
//     of 16-row fragments. Two workgroups per CU fit at D=128.
//   - A wave's vector work runs under its own products: the maximum of a
//     tile's scores under the first half of the next tile's, its weights
//     under the second half and under the results of the weights before them
//     (one after the other, two waves a SIMD: matrix cores 42 % and vector ALU
//     46 % of the cycles, hardly any at once; now 55 and 52 %). Scheduling
//     barriers pin the order; other shares of products a group, 3 to 8 fragments
//     read ahead and wave priorities measured the same.
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
//   - K and V have two places each in LDS and are filled straight from the
//     cache (8-bit ones by way of registers, which widen): V a tile ahead, K
//     two, one barrier per tile.
//   - Tiles are taken in pairs, so that scores stay in the registers where
//     they were formed. Of an even number the last takes scores that nobody
//     asked for with it; forms of their own for it needed scratch and made
//     short prompts wait for code (8192 tokens 552 us, 64 short ones 57).
//   - The 16-bit weights are summed as they are rounded (one dot product
//     instruction a pair), so that their rounding cancels in the quotient,
//     and the row's largest weight is exactly one: accumulators are
//     rescaled whenever a maximum moves. Letting it grow by 2^8 first
//     would save 3 % and raise the distance to 64-bit results by 2 to 7 %
//     (now 1 % below that of unrounded sums).
//   - Results are stored 16 B a lane.
// Scores, weights and results one after the other -> so, us, 32/8 heads of
// 128: one prompt of 8192 tokens 615 -> 527 (1.04 PFLOP/s), with an 8-bit cache
// 599 -> 551; 2048 63 -> 52; 512 after 1536 to 15872, 4 such 410 -> 312; 64 of
// 33..223 48.7 -> 44.6; 4 x 2048 tokens, 16/8 heads of 256, 284 -> 211.
//
// Role of the reference's triton_unified_attention.py:179 (prefill side)
// and prefix_prefill.py.

#pragma once

#include <type_traits>

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
// Workgroups that a CU is to hold, by registers. Three with heads of 64: an
// 8-bit cache left to itself takes two registers too many for that, and short
// prompts wait for a second round (53 of 124 tokens, 32/4 heads 25.1 us, so
// 21.6; 23 of 107, 32/8 heads 12.0 and 10.5). Four spill (1.25 to 1.4 times).
template <int HD>
constexpr int pf_per_cu = HD == 256 ? 1 : HD == 64 ? 3 : 2;

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
  auto block_of = [&](int kt) { return load_uniform(bt + min(kt, kt_end - 1)); };

  // A tile of keys (PLANE 0) or values (1) on its way to a place in LDS: fills,
  // or, where it has to be widened, registers until land().
  i32x4 kv_reg[2][FP8 ? LD : 1];
  auto fetch = [&](auto plane, int phys, int place) {
    constexpr int PLANE = decltype(plane)::value;
    const elem* src = a.kv_cache + PLANE * kv_plane_stride +
                      ((int64_t)phys * num_kv_heads + kvh) * TILE;
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      if constexpr (FP8)
        kv_reg[PLANE][i] = *reinterpret_cast<const i32x4*>(
            src + (i * PF_BLOCK + threadIdx.x) * EPV);
      else {
        // What lies in LDS where this lane's 16 B land.
        constexpr int ROWS = PF_BLOCK * 8 / HD;   // of a piece
        const int r = threadIdx.x * 8 / HD, c = threadIdx.x * 8 % HD / 8;
        const int at = PLANE == 0 ? k_chunk<HD>(i * ROWS + r, c) * 8
                                  : v_seg<HD>(i * ROWS + r, c >> 1) * 16 +
                                        (c & 1) * 8;
        lds_fill16(src + i * PF_BLOCK * EPV, (uint32_t)(r * HD + at) * 2,
                   lds + (PLANE * 2 + place) * TILE * 2 +
                       (i * PF_BLOCK + wave * WAVE_SIZE) * 16);
      }
    }
  };
  auto land = [&](auto plane, int kt, int place) {
    constexpr int PLANE = decltype(plane)::value;
    // Values of rows no token has been written to yet may hold anything, and
    // their zero weight does not stop a NaN.
    const bool edge = PLANE == 1 && kt * KVTILE + KVTILE > ctx;
    short* to = reinterpret_cast<short*>(lds) + (PLANE * 2 + place) * TILE;
    if constexpr (FP8) {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const int e = (i * PF_BLOCK + threadIdx.x) * EPV;
        const int r = e / HD;
        const int c = (e % HD) / 8;
        i32x4 v = kv_reg[PLANE][i];
        if (edge) {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = kt * KVTILE + r < ctx ? v[j] : 0;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int2 x = fp8x4_widen<Tag>(v[h * 2]);
          const int2 y = fp8x4_widen<Tag>(v[h * 2 + 1]);
          const int at = PLANE == 0 ? k_chunk<HD>(r, c + h) * 8
                                    : v_seg<HD>(r, (c + h) >> 1) * 16 +
                                          ((c + h) & 1) * 8;
          *reinterpret_cast<i32x4*>(to + r * HD + at) =
              i32x4{x.x, x.y, y.x, y.y};
        }
      }
    } else if (edge) {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const int e = (i * PF_BLOCK + threadIdx.x) * EPV;
        if (kt * KVTILE + e / HD >= ctx)
          *reinterpret_cast<i32x4*>(to + e) = i32x4{0, 0, 0, 0};
      }
    }
  };
  // All fills of this wave have landed (what follows stays behind them).
  auto landed = [&] {
    if constexpr (!FP8) {
      lds_fill_wait();
      asm volatile("" ::: "memory");
    }
  };
  constexpr std::integral_constant<int, 0> KEYS{};
  constexpr std::integral_constant<int, 1> VALUES{};

  // Products of a step in their order: the first and the second 32 keys of the
  // next tile's scores, then the four chunks of 16 keys of this one's results.
  constexpr int QK = 2 * KF, ALL = QK + 4 * DS;
  // Fragments read ahead (with a fourth there would be scratch for these).
  constexpr int AHEAD = FP8 && HD == 64 ? 3 : 4;
  int k_at[KF], v_at[DS];   // first fragments of a tile, in its bytes
#pragma unroll
  for (int kk = 0; kk < KF; ++kk)
    k_at[kk] = (l32 * HD + k_chunk<HD>(l32, kk * 2 + half) * 8) * 2;
#pragma unroll
  for (int i = 0; i < DS; ++i) {
    const int r = half * 4 + ((lane & 15) >> 2);
    v_at[i] = (r * HD + v_seg<HD>(r, i * 2 + ((lane >> 4) & 1)) * 16 +
               (lane & 3) * 4) * 2;
  }
  auto fragment = [&](int m, int k_place, int v_place) -> s16x8 {
    if (m < QK)   // (the moves of rows 16 and 32 apart are the same)
      return *reinterpret_cast<const s16x8*>(
          lds + k_place * TILE * 2 + m / KF * 32 * HD * 2 + k_at[m % KF]);
    const char* v = lds + (2 + v_place) * TILE * 2 +
                    (m - QK) / DS * 16 * HD * 2 + v_at[(m - QK) % DS];
    const s16x4 c0 = lds_read_tr(v), c1 = lds_read_tr(v + 8 * HD * 2);
    return __builtin_shufflevector(c0, c1, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  const f32x16 zero = {};
  const int first = block_of(kt0);
  int next = block_of(kt0 + 1), second = block_of(kt0 + 2);

  // One tile: its scores s become weights and results, between the products of
  // the next one's scores t (MORE; where there is none, of what lies there).
  auto tile_step = [&](const int kt, f32x16 (&s)[2], f32x16 (&t)[2],
                       const int place, auto more) {
    constexpr bool MORE = decltype(more)::value;
    constexpr int FIRST = MORE ? 0 : QK;
    if constexpr (MORE) {
      // (Of either place the last read lies before the barrier.)
      if (kt + 1 < kt_end) fetch(VALUES, next, 1 - place);
      if (kt + 2 < kt_end) fetch(KEYS, second, place);
      next = second;
      second = block_of(kt + 3);
    }
    s16x8 frag[AHEAD], pf[4];
    auto read = [&](int m) {
      if (m >= FIRST && m < ALL)
        frag[m % AHEAD] = fragment(m, 1 - place, place);
    };
    auto product = [&](int m) {
      if (m < QK)
        t[m / KF] = mfma32<Tag>(frag[m % AHEAD], qf[m % KF],
                                m % KF == 0 ? zero : t[m / KF]);
      else
        o[(m - QK) % DS] = mfma32<Tag>(frag[m % AHEAD], pf[(m - QK) / DS],
                                       o[(m - QK) % DS]);
      read(m + AHEAD);
    };
    // --- mask, only where the tile meets an edge -------------------------
    // Register r of subtile n is key n*32 + 8*(r/4) + 4*half + r%4.
    const int key_base = kt * KVTILE + half * 4;
    if (kt * KVTILE + KVTILE - 1 > first_pos ||
        (sliding_window > 0 && kt * KVTILE <= last_pos - sliding_window)) {
      const int hi = qpos - key_base;
      const int lo = sliding_window > 0 ? hi - sliding_window : -1;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = n * 32 + 8 * (r >> 2) + (r & 3);
          s[n][r] = key <= hi && key > lo ? s[n][r] : PF_NEG;
        }
    }
#pragma unroll
    for (int m = FIRST; m < FIRST + AHEAD; ++m) read(m);

    // --- running softmax --------------------------------------------------
    // med3 with +inf is a maximum that the compiler fuses in threes (fmaxf
    // first quiets each score: 37 more instructions a tile, 2 %).
    float mx = PF_NEG;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = g * 2; r < g * 2 + 2; ++r) {
        mx = __builtin_amdgcn_fmed3f(mx, s[0][r], INFINITY);
        mx = __builtin_amdgcn_fmed3f(mx, s[1][r], INFINITY);
      }
      if constexpr (MORE) {
#pragma unroll
        for (int m = KF * g / 8; m < KF * (g + 1) / 8; ++m) product(m);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
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

    // --- weights, and O^T += V^T P^T ---------------------------------------
    // Half a chunk of weights a group, then as many products as weights are
    // there for.
    constexpr int TO[9] = {8, 11, 14, 17, 20, 22, 24, 26, 28};
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      __builtin_amdgcn_sched_barrier(0);
      const int c = g / 2;
      i32x4 pk = g % 2 ? __builtin_bit_cast(i32x4, pf[c]) : i32x4{};
#pragma unroll
      for (int j = g % 2 * 2; j < g % 2 * 2 + 2; ++j) {
        const int r = (c & 1) * 8 + j * 2;
        const float p0 = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[c >> 1][r], scale_log2, shift));
        const float p1 = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[c >> 1][r + 1], scale_log2, shift));
        pk[j] = pack2<Tag>(p0, p1);
        l_run = add_pair<Tag>(pk[j], l_run);
      }
      pf[c] = __builtin_bit_cast(s16x8, pk);
      const int m0 = TO[g] * KF / 8, m1 = TO[g + 1] * KF / 8;
#pragma unroll
      for (int m = m0; m < m1; ++m)
        if (m >= FIRST) product(m);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = TO[8] * KF / 8; m < ALL; ++m) product(m);
    if constexpr (MORE) {
      landed();
      if (kt + 1 < kt_end) land(VALUES, kt + 1, 1 - place);
      if (kt + 2 < kt_end) land(KEYS, kt + 2, place);
    }
    lds_barrier();
  };

  fetch(KEYS, first, 0);
  fetch(VALUES, first, 0);
  if (!FP8 && kt0 + 1 < kt_end) fetch(KEYS, next, 1);
  landed();
  land(KEYS, kt0, 0);
  land(VALUES, kt0, 0);
  if (FP8 && kt0 + 1 < kt_end) fetch(KEYS, next, 1);
  lds_barrier();
  f32x16 sa[2], sb[2];
#pragma unroll
  for (int m = 0; m < QK; ++m)
    sa[m / KF] = mfma32<Tag>(fragment(m, 0, 0), qf[m % KF],
                             m % KF == 0 ? zero : sa[m / KF]);
  if (FP8 && kt0 + 1 < kt_end) land(KEYS, kt0 + 1, 1);
  lds_barrier();   // the first keys' place is free
  int kt = kt0;
#pragma unroll 1
  for (; kt + 1 < kt_end; kt += 2) {
    tile_step(kt, sa, sb, 0, std::true_type{});
    tile_step(kt + 1, sb, sa, 1, std::true_type{});
  }
  if (kt < kt_end) tile_step(kt, sa, sb, 0, std::false_type{});

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
