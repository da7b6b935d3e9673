// Paged decode attention for MI355X (gfx950, CDNA4): the work of a workgroup
// (kernels: attention_decode.hip, and attention_mixed.hip beside prompts).
//
// What bounds it: one pass over the cached keys and values. At 2..16
// flops per byte everything else only has to stay out of the way of the
// loads, so the kernel keeps as many bytes in flight as registers allow
// and spends few issue slots per byte:
//   - A wave owns 32 keys at a time (16 where rows are 512 B) and never
//     meets another wave before the end, so there is no barrier in the
//     loop. The next keys are loaded as soon as the registers of the
//     current ones are free.
//   - Scores are S^T = K Q^T on the matrix cores: a K row goes from HBM
//     straight into the A fragment (16 B per lane), the query heads of
//     the group are the columns. No long cross-lane sum per key and head,
//     which is what the vector-ALU form of this kernel spent its time on.
//   - A group has at most 8 of the 16 columns. The other 8 hold the second
//     half of the queries' columns, and two neighbouring rows of the
//     fragment the halves of one key: the same products, but a load takes
//     whole lines of 8 keys instead of half lines of 16, and a score is the
//     sum of two lanes (one rotation). us, half lines and whole, marked as
//     below: keys that no cache holds, 32 x 4096 keys 108 and 91, 64 x 4096 221
//     and 179, 1 x 1000 8.7 and 8.2, 16 x 128 6.2 and 5.3, 4 x 20 4.44 and
//     4.46; keys that the last-level cache may hold in part, 256 x 129..2176
//     210 and 203, 64 x 4096..8192 with an 8-bit cache 147 and 145, 32 x 4096
//     87 either way. By quarters of a group of 4 no faster. What a window of
//     1024 keys reads again and again from the last-level cache is 8 % slower
//     (119 x 5600, 28/4 heads 44 and 48; from memory 80 and 56), rows of up to
//     60 keys in L2 0.1 us.
//   - O^T = V^T P^T: V passes through this wave's own LDS slice to be
//     transposed on the read. The lane that holds the scores of keys
//     (4g..4g+3, 16+4g..) holds exactly the P^T fragment of those keys
//     when the contraction runs over keys in that order, so P never
//     moves between lanes.
//   - Keys and values are read as lines that leave L2 first: each is needed
//     once, and they no longer push out what other workgroups are about to
//     read. (Rows that have most of their keys in common: 64 x 2000 keys, 1920
//     of them common, 32 heads ungrouped, 135 us; half lines of keys, which had
//     to stay in L2 for the other half, 164, and nothing marked 147.) Where a
//     wave is a row of few keys, keys are not marked: what a step holds past
//     the row's end repeats its last key (200 x 1..60 keys 9.8 us, marked
//     10.2).
//   - P stays at more than 16 bits: it is split in two 16-bit parts
//     (p = hi + lo, error 2^-17) and multiplied twice; the matrix cores
//     are idle here anyway. Sums and outputs are fp32. Results are as far
//     from 64 bits as with fp32 weights, to six digits (1.64328e-3 at 1 x
//     1000 keys, 1.66106e-3 at 1024 x 129..176, fp16 2.07694e-4 at 40 x
//     100..4000).
// Against the vector-ALU form it replaced (16 lanes per token, dot
// products reduced with shuffles), us per layer at 32 query and 8 KV
// heads of 128:
//   1 x 1000 keys 46 -> 8; 256 x 129..2176 keys 349 -> 203 (6.0 TB/s);
//   1024 x 129..176 keys 206 -> 108 (132 with the last 32 keys of a row read
//   whole), 118 between the other work of a model's layer; 16 x 4096 keys 46;
//   64 x 4096..8192 keys, fp8 cache 371 -> 145.
//
// The KV cache layout [2, blocks, kv_heads, block_size=64, D] keeps each
// (block, head) tile contiguous (16 KB at D=128).
//
// Role of the reference's paged_attention (csrc/rocm/attention.cu:321,1420).

#pragma once

#include "arrivals.h"
#include "common.h"

namespace vllm_amd {

constexpr int DEC_WAVES = 4;
constexpr int DEC_BLOCK = DEC_WAVES * WAVE_SIZE;
constexpr int DEC_KEYS = 32;    // keys per wave and step, at most
constexpr int MAX_GROUP = 8;    // query heads per KV head
constexpr int MAX_PARTS = 64;   // partitions of a row: lanes of a wave
constexpr float DEC_NEG = -3.0e38f;
constexpr float DEC_LOG2E = 1.4426950408889634f;

// Bytes of a V row are moved in 32 B segments (16 columns, what one
// transposing read takes from a row). Rotating the segments by the row
// spreads the rows a read touches over all 64 banks.
template <int HD> DEVINL int v_slot(int row, int seg) {
  if constexpr (HD == 64) return seg ^ ((row >> 1) & 3);
  return seg ^ (row & 7);
}

// Keys per wave and step. 32 rows of 512 B each for keys and values, the
// queries and 16 x 256 outputs are more registers than the two workgroups
// of a CU have (340; one workgroup then, values moved between register
// files): 16 a step instead takes 228. us: 16 x 750..1500 keys, 16 KV heads
// 58 -> 53, 64 x 300..3000 (4) 102 -> 98, 256 x 150..300 through a window of
// 128 (16, three query heads each) 146 -> 102. At 128 columns 16 keys are no
// faster for long rows (256 x 129..2176 228 -> 231).
template <typename CTag, int HD>
constexpr int dec_keys =
    HD == 256 && sizeof(typename CacheTraits<CTag>::elem) == 2 ? 16
                                                               : DEC_KEYS;

// Parts of a key row that lie on neighbouring lanes: one load of 16 / S rows
// then takes whole lines of 128 B. (A row of 64 B is taken whole as it is.)
// Where a wave is a row and the cache has 8 bits, half lines are ahead: a step
// of 32 keys is one load a lane either way, and the sums of two lanes come on
// top (us, whole and half lines, 16/8 heads: 600 rows x 1..350 keys 53.3 and
// 47.7, from HBM 74 and 71; 1000 x 1..120 the same).
template <typename CTag, int HD, int WPR>
constexpr int dec_split =
    HD * sizeof(typename CacheTraits<CTag>::elem) >= 128 &&
            (WPR > 1 || sizeof(typename CacheTraits<CTag>::elem) == 2)
        ? 2
        : 1;

// First key this row attends, rounded down so that a wave's 32 keys
// never leave a cache block.
DEVINL int dec_base(int ctx, int window) {
  return window > 0 ? (max(0, ctx - window) & ~(DEC_KEYS - 1)) : 0;
}

// WPR 4: one workgroup is (kv head, decode row, partition of part_len
// keys) and a wave takes every fourth step of them. WPR 1: a wave is a row
// of its own, whole, for batches of short rows. A row of several partitions
// (only where not WHOLE) leaves fp32 partials with their running maximum
// (log2 domain) and sum; the last of its workgroups to arrive merges them.
// (With a second launch for that: 1 x 1000 keys 9.4 us, now 7.8; 4 x 8192 32.4,
// now 27.3.)
template <typename CTag> struct DecodeArgs {
  short* out;            // [Tdec, Hq, D] (16-bit)
  float* tmp_out;        // [Tdec, Hq, parts, D]
  float* tmp_lse;        // [Tdec, Hq, parts, 2]
  unsigned* arrived;     // [Tdec, Hkv]
  const short* q;        // [Tdec, Hq, D]
  const typename CacheTraits<CTag>::elem* kv_cache;  // [2, blocks, Hkv, 64, D]
  const int* block_table;   // [num_reqs, max_blocks]
  const int* seq_lens;      // [num_reqs]
  float scale_log2;
  int group, num_kv_heads, num_seqs, max_blocks_per_req, num_parts, part_len;
  int64_t kv_plane_stride;  // elements between K and V planes
  int64_t q_stride;         // elements between q token rows
  int sliding_window;
};

// Bytes of LDS of a workgroup: V slices of the waves, or what the waves
// (group <= 8 of the 16 columns) and the partitions merge there at the end.
constexpr int dec_merge(int hd) { return DEC_WAVES * MAX_GROUP * (hd * 4 + 8); }
template <typename CTag, int HD>
constexpr int dec_lds = DEC_WAVES * dec_keys<CTag, HD> * HD * 2 >
                                dec_merge(HD)
                            ? DEC_WAVES * dec_keys<CTag, HD> * HD * 2
                            : dec_merge(HD);

template <typename Tag, typename CTag, bool WHOLE, int HD, int WPR>
DEVINL void decode_rows(const DecodeArgs<CTag>& a, const int kvh,
                        const int row_block, const int part_block,
                        char* lds) {
  static_assert(WPR == DEC_WAVES || (WPR == 1 && WHOLE));
  using elem = typename CacheTraits<CTag>::elem;
  constexpr bool FP8 = sizeof(elem) == 1;
  constexpr int EPV = 16 / sizeof(elem);          // elements per 16 B
  constexpr int KEYS = dec_keys<CTag, HD>;
  constexpr int KT = KEYS / 16;                   // score tiles
  constexpr int KF = HD / 32;                     // MFMA steps over D
  constexpr int S = dec_split<CTag, HD, WPR>;
  static_assert(MAX_GROUP * S <= 16);
  constexpr int NT = KT * S;                      // loaded tiles of 16 / S keys
  constexpr int KN = HD * (int)sizeof(elem) / 64 / S;   // 16 B K loads of one
  constexpr int QF = KF / S;                      // fragments of the queries
  constexpr int KR = 4 / S;                       // keys of a lane in a tile
  constexpr int VN = KEYS * HD / EPV / WAVE_SIZE;
  constexpr int DS = HD / 16;                     // output column tiles
  constexpr int V_BYTES = KEYS * HD * 2;          // per wave

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  short* __restrict__ const out = a.out;
  float* __restrict__ const tmp_out = a.tmp_out;
  float* __restrict__ const tmp_lse = a.tmp_lse;
  const elem* __restrict__ const kv_cache = a.kv_cache;
  const int group = a.group, num_kv_heads = a.num_kv_heads;
  const int num_parts = a.num_parts, part_len = a.part_len;
  const int64_t kv_plane_stride = a.kv_plane_stride;
  const int sliding_window = a.sliding_window;
  const float scale_log2 = a.scale_log2;
  // Decode row == request row.
  const int seq = WPR > 1 ? row_block : row_block * DEC_WAVES + wave;
  if (WPR == 1 && seq >= a.num_seqs) return;   // (no barrier below then)
  const int part = WPR > 1 ? part_block : 0;
  const int ctx = load_uniform(a.seq_lens + seq);
  const int num_q_heads = num_kv_heads * group;
  const int hq0 = kvh * group;
  const int t_lo = sliding_window > 0 ? max(0, ctx - sliding_window) : 0;
  const int t_first = dec_base(ctx, sliding_window);
  const int t_begin = t_first + part * part_len;
  const int t_end = min(ctx, t_begin + part_len);
  // Partitions of this row that hold keys.
  const int used =
      WHOLE ? 1 : min(num_parts, (ctx - t_first + part_len - 1) / part_len);

  if (t_begin >= t_end) {
    if (part == 0)   // a row without keys (padding) is zero
      for (int e = WPR > 1 ? threadIdx.x : lane; e < group * HD;
           e += WPR * WAVE_SIZE)
        out[((int64_t)seq * num_q_heads + hq0) * HD + e] = 0;
    return;
  }

  const int l16 = lane & 15;
  const int l4 = lane >> 4;

  char* v_lds = lds + wave * V_BYTES;

  // B fragments of the queries: column h + 16 / S * part is that part of the
  // columns of head h of the group (of head 0 where the group ends before).
  const int part_q = l16 / (16 / S);
  s16x8 qf[QF];
  {
    const int h = l16 % (16 / S);
    const short* qb = a.q + (int64_t)seq * a.q_stride +
                      (int64_t)(hq0 + (h < group ? h : 0)) * HD;
#pragma unroll
    for (int kk = 0; kk < QF; ++kk) {
      // With an fp8 cache a 16 B load is two fragments' worth of one row.
      constexpr int PER = FP8 ? 2 : 1;
      const int d =
          ((kk / PER * 4 + l4) * S + part_q) * EPV + kk % PER * 8;
      qf[kk] = *reinterpret_cast<const s16x8*>(qb + d);
    }
  }

  const int* bt = a.block_table + (int64_t)seq * a.max_blocks_per_req;
  auto tile_of = [&](int key0) {
    return kv_cache +
           ((int64_t)load_uniform(bt + (key0 >> 6)) * num_kv_heads + kvh) *
               (64 * HD) +
           (key0 & 63) * HD;
  };
  // Row l16 of tile t is part l16 % S of key k_row(t): a lane ends up with
  // the scores of keys 16 * T + 4 * l4 + 0..3 however they are loaded.
  auto k_row = [&](int t) {
    const int p = l16 / S;
    return t / S * 16 + p / KR * 4 + t % S * KR + p % KR;
  };
  i32x4 kr[NT][KN], vr[VN];
  // Rows of a step that the row does not attend repeat the nearest one it
  // does: they cost no bytes.
  auto load_k = [&](const elem* tile, int key0) {
    const int lo = t_lo - key0, hi = t_end - 1 - key0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int r = min(max(k_row(t), lo), hi);
#pragma unroll
      for (int i = 0; i < KN; ++i) {
        const i32x4* at = reinterpret_cast<const i32x4*>(
            tile + r * HD + ((i * 4 + l4) * S + l16 % S) * EPV);
        kr[t][i] = WPR > 1 ? __builtin_nontemporal_load(at) : *at;
      }
    }
  };
  auto load_v = [&](const elem* tile, int key0) {
    const int lo = t_lo - key0, hi = t_end - 1 - key0;
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const int e = (i * WAVE_SIZE + lane) * EPV;
      const int r = min(max(e / HD, lo), hi);
      vr[i] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(
          tile + kv_plane_stride + r * HD + e % HD));
    }
  };

  float m_run = DEC_NEG, l_run = 0.f;   // of head l16; l: this lane's keys
  f32x4 o[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // One step of KEYS keys; with NEXT the loads of the wave's next ones are
  // issued as the registers become free (a template flag and not a test
  // inside, so that the waits count exactly the older loads).
  constexpr int STRIDE = WPR * KEYS;
  auto step = [&](int key0, auto has_next) {
    constexpr bool NEXT = decltype(has_next)::value;
    const elem* next_tile =
        NEXT ? tile_of(key0 + STRIDE) : nullptr;
    // ---- S^T: rows are keys, columns heads -----------------------------
    f32x4 s[KT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < QF; ++kk) {
        s16x8 f;
        if constexpr (FP8) {
          const i32x4 r = kr[t][kk >> 1];
          const int2 x = fp8x4_widen<Tag>(r[(kk & 1) * 2]);
          const int2 y = fp8x4_widen<Tag>(r[(kk & 1) * 2 + 1]);
          f = __builtin_bit_cast(s16x8, (i32x4){x.x, x.y, y.x, y.y});
        } else {
          f = __builtin_bit_cast(s16x8, kr[t][kk]);
        }
        c = mfma16<Tag>(f, qf[kk], c);
      }
      // Of each key the part that met its own columns; then the others'.
#pragma unroll
      for (int j = 0; j < KR; ++j) {
        float y = c[j * S];
        if constexpr (S == 2) y = part_q == 0 ? y : c[j * S + 1];
        if constexpr (S == 2) y += row_ror<8>(y);
        s[t / S][t % S * KR + j] = y;
      }
    }
    if constexpr (NEXT) load_k(next_tile, key0 + STRIDE);

    // ---- V to LDS, rows outside [t_lo, t_end) as zeros ------------------
    // (a stale cache row may hold anything, and 0 * NaN is NaN).
    const bool edge = key0 < t_lo || key0 + KEYS > t_end;
    if (edge) {
#pragma unroll
      for (int i = 0; i < VN; ++i) {
        const int key = key0 + (i * WAVE_SIZE + lane) * EPV / HD;
        const bool in = (key >= t_lo) & (key < t_end);
#pragma unroll
        for (int j = 0; j < 4; ++j) vr[i][j] = in ? vr[i][j] : 0;
      }
    }
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const int e = (i * WAVE_SIZE + lane) * EPV;
      const int row = e / HD;
      const i32x4 v = vr[i];
      const int c16 = (e % HD) / 8;   // 16 B chunk of the 16-bit row
      char* dst = v_lds + row * (HD * 2) + v_slot<HD>(row, c16 >> 1) * 32;
      if constexpr (FP8) {
        const int2 a = fp8x4_widen<Tag>(v[0]), b = fp8x4_widen<Tag>(v[1]);
        const int2 c = fp8x4_widen<Tag>(v[2]), d = fp8x4_widen<Tag>(v[3]);
        i32x4* p = reinterpret_cast<i32x4*>(dst);
        p[0] = i32x4{a.x, a.y, b.x, b.y};
        p[1] = i32x4{c.x, c.y, d.x, d.y};
      } else {
        *reinterpret_cast<i32x4*>(dst + (c16 & 1) * 16) = v;
      }
    }
    if constexpr (NEXT) load_v(next_tile, key0 + STRIDE);

    // ---- running softmax, log2 domain ----------------------------------
    // A key outside the row's range scores DEC_NEG and weighs nothing
    // even where the whole step is outside it.
    bool in[KT][4];
    float mx = DEC_NEG;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = key0 + t * 16 + l4 * 4 + r;
        in[t][r] = (key >= t_lo) & (key < t_end);
        s[t][r] = in[t][r] ? s[t][r] * scale_log2 : DEC_NEG;
        mx = fmaxf(mx, s[t][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx);
    if (__any(m_new > m_run)) {
      const float f = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= f;
#pragma unroll
      for (int i = 0; i < DS; ++i) o[i] *= f;
      m_run = m_new;
    }
    i32x4 hi = {0, 0, 0, 0}, lo = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        const float e0 = __builtin_amdgcn_exp2f(s[t][r] - m_run);
        const float e1 = __builtin_amdgcn_exp2f(s[t][r + 1] - m_run);
        const float p0 = in[t][r] ? e0 : 0.f;
        const float p1 = in[t][r + 1] ? e1 : 0.f;
        l_run += p0 + p1;
        const int h = pack2<Tag>(p0, p1);
        hi[t * 2 + r / 2] = h;
        lo[t * 2 + r / 2] =
            pack2<Tag>(p0 - unpack_lo<Tag>(h), p1 - unpack_hi<Tag>(h));
      }
    const s16x8 p_hi = __builtin_bit_cast(s16x8, hi);
    const s16x8 p_lo = __builtin_bit_cast(s16x8, lo);

    // ---- O^T += V^T P^T -------------------------------------------------
    // LDS operations of one wave complete in order; the fences only keep
    // the compiler from moving them.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int row = l4 * 4 + (l16 >> 2);
#pragma unroll
    for (int i = 0; i < DS; ++i) {
      const int off = (l16 & 3) * 8;
      const s16x4 a = lds_read_tr(v_lds + row * (HD * 2) +
                                  v_slot<HD>(row, i) * 32 + off);
      if constexpr (KT == 1) {
        o[i] = mfma16<Tag>(a, __builtin_shufflevector(p_lo, p_lo, 0, 1, 2, 3),
                           o[i]);
        o[i] = mfma16<Tag>(a, __builtin_shufflevector(p_hi, p_hi, 0, 1, 2, 3),
                           o[i]);
        continue;
      }
      const s16x4 b = lds_read_tr(v_lds + (row + 16) * (HD * 2) +
                                  v_slot<HD>(row + 16, i) * 32 + off);
      const s16x8 v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
      o[i] = mfma16<Tag>(v, p_lo, o[i]);
      o[i] = mfma16<Tag>(v, p_hi, o[i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  int key0 = t_begin + (WPR > 1 ? wave * KEYS : 0);
  if (key0 < t_end) {
    const elem* tile = tile_of(key0);
    load_k(tile, key0);
    load_v(tile, key0);
    for (; key0 + STRIDE < t_end; key0 += STRIDE)
      step(key0, std::true_type{});
    step(key0, std::false_type{});
  }

  // ---- merge the waves ----------------------------------------------------
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if constexpr (WPR == 1) {   // nothing to merge
    const float inv_l = l_run > 0.f || l_run != l_run ? 1.f / l_run : 0.f;
    if (l16 < group) {
      short* ob =
          out + ((int64_t)seq * num_q_heads + hq0 + l16) * HD + l4 * 4;
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        int2 v;
        v.x = pack2<Tag>(o[i][0] * inv_l, o[i][1] * inv_l);
        v.y = pack2<Tag>(o[i][2] * inv_l, o[i][3] * inv_l);
        *reinterpret_cast<int2*>(ob + i * 16) = v;
      }
    }
    return;
  }
  __syncthreads();   // every wave is done with its V slice
  float* o_red = reinterpret_cast<float*>(lds);  // [wave][MAX_GROUP][HD]
  // [wave][MAX_GROUP]: maximum and sum
  auto* ml_red = reinterpret_cast<float(*)[MAX_GROUP][2]>(
      lds + DEC_WAVES * MAX_GROUP * HD * 4);
  if (l16 < group) {
#pragma unroll
    for (int i = 0; i < DS; ++i)
      *reinterpret_cast<f32x4*>(
          o_red + (wave * MAX_GROUP + l16) * HD + i * 16 + l4 * 4) = o[i];
    if (l4 == 0) {
      ml_red[wave][l16][0] = m_run;
      ml_red[wave][l16][1] = l_run;
    }
  }
  __syncthreads();
  auto store4 = [&](int g, int d, f32x4 v) {
    *reinterpret_cast<int2*>(
        out + ((int64_t)seq * num_q_heads + hq0 + g) * HD + d) =
        int2{pack2<Tag>(v[0], v[1]), pack2<Tag>(v[2], v[3])};
  };
  for (int e = threadIdx.x * 4; e < group * HD; e += DEC_BLOCK * 4) {
    const int g = e / HD;
    const int d = e % HD;
    float M = DEC_NEG;
#pragma unroll
    for (int w = 0; w < DEC_WAVES; ++w) M = fmaxf(M, ml_red[w][g][0]);
    float L = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < DEC_WAVES; ++w) {
      const float c = __builtin_amdgcn_exp2f(ml_red[w][g][0] - M);
      L += ml_red[w][g][1] * c;
      acc += *reinterpret_cast<const f32x4*>(
                 o_red + (w * MAX_GROUP + g) * HD + d) *
             c;
    }
    if (WHOLE || used == 1) {
      store4(g, d, acc * (L > 0.f || L != L ? 1.f / L : 0.f));
    } else {
      const int64_t row =
          ((int64_t)seq * num_q_heads + hq0 + g) * num_parts + part;
      part_put(reinterpret_cast<f32x4*>(tmp_out + row * HD + d), acc);
      if (d == 0) {
        part_put(tmp_lse + row * 2, M);
        part_put(tmp_lse + row * 2 + 1, L);
      }
    }
  }
  if constexpr (!WHOLE) {
    // ---- merge the partitions: sum_p o_p 2^(m_p - M) / sum_p l_p 2^(m_p -
    // M), the weights of each head in LDS ----------------------------------
    if (used == 1) return;
    float* w_lds = reinterpret_cast<float*>(lds);   // [group][MAX_PARTS]
    static_assert(MAX_GROUP * MAX_PARTS * 4 + 4 <= dec_lds<CTag, HD>);
    if (!last_to_arrive(
            a.arrived, (int64_t)seq * num_kv_heads + kvh, used,
            reinterpret_cast<unsigned*>(w_lds + MAX_GROUP * MAX_PARTS)))
      return;
    const int64_t row0 = ((int64_t)seq * num_q_heads + hq0) * num_parts;
    // Parts come from beyond L2: all that a thread needs is on its way at
    // once, weights and the first eight partitions of its columns.
    constexpr int AT_ONCE = 8;
    f32x4 first[AT_ONCE];
    const int e0 = threadIdx.x * 4;
    auto part_of = [&](int e, int p) {
      return reinterpret_cast<const f32x4*>(
          tmp_out + (row0 + (int64_t)(e / HD) * num_parts + p) * HD + e % HD);
    };
#pragma unroll
    for (int p = 0; p < AT_ONCE; ++p)
      if (e0 < group * HD && p < used) first[p] = part_get(part_of(e0, p));
    constexpr int HEADS = MAX_GROUP / DEC_WAVES;
    float m[HEADS], l[HEADS];
#pragma unroll
    for (int i = 0; i < HEADS; ++i) {   // lane p: partition p
      const int g = wave + i * DEC_WAVES;
      const bool in = g < group && lane < used;
      const float* lse = tmp_lse + (row0 + (int64_t)g * num_parts + lane) * 2;
      m[i] = in ? part_get(lse) : DEC_NEG;
      l[i] = in ? part_get(lse + 1) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < HEADS; ++i) {
      const float w = __builtin_amdgcn_exp2f(m[i] - wave_reduce_max(m[i]));
      const float L = wave_reduce_sum(l[i] * w);
      w_lds[(wave + i * DEC_WAVES) * MAX_PARTS + lane] =
          L > 0.f || L != L ? w * (1.f / L) : 0.f;
    }
    __syncthreads();
    for (int e = e0; e < group * HD; e += DEC_BLOCK * 4) {
      const float* w = w_lds + e / HD * MAX_PARTS;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      for (int p0 = 0; p0 < used; p0 += AT_ONCE) {
        // Reads past the last partition repeat it: with a branch each waits
        // for the one before (16/2 heads of 256, 3 x 2916 keys 19.5 us, now
        // 15.4).
        f32x4 v[AT_ONCE];
        if (e == e0 && p0 == 0) {
#pragma unroll
          for (int i = 0; i < AT_ONCE; ++i) v[i] = first[i];
        } else {
#pragma unroll
          for (int i = 0; i < AT_ONCE; ++i)
            v[i] = part_get(part_of(e, min(p0 + i, used - 1)));
        }
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i)
          if (p0 + i < used) acc += v[i] * w[p0 + i];
      }
      store4(e / HD, e % HD, acc);
    }
  }
}

}  // namespace vllm_amd
