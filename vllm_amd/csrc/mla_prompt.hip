// MLA attention of prompt portions per head, for CDNA4 (gfx950).
//
// In the latent space a (query, key) pair costs 576 + 512 products a head;
// with keys and values carried out of it (K = c W_UK^T, V = c W_UV, 128
// wide each) it costs 192 + 128, and carrying them out costs as much per
// context token as carrying a query in and its result out. So portions of
// many tokens take this form:
//   mla_expand_kernel   keys, values and rotary parts of each request's
//                       context, from the paged latent cache, per head
//   mla_prompt_kernel   causal attention over them
// Values are rounded to the cache's type, as results are in the latent
// form; weights keep more than 16 bits (hi + lo). Keys are fp16 for a bf16
// cache too: in sharp softmaxes the 128 roundings of a key weigh more than
// the 512 of a query carried into the latent space. 5 prompts of 283 tokens,
// queries of deviation 1 / 4 / 8, distance to 64 bits in thousandths: keys in
// bf16 2.36 / 3.11 / 3.68, the latent form 2.37 / 3.08 / 3.61, keys in fp16
// 2.27 / 2.34 / 2.36 (fp16 products run 2 % slower, power bound); with an
// fp16 cache 0.295 / 0.389 / 0.460, the latent form 0.296 / 0.385 / 0.451.
// So that no key leaves fp16's range, 64 tokens x 64 columns share a power of
// two, which is one unless their largest is below 1/4 or from 2^15.
// 128 heads, prompts of 300, 1300 and 2301 tokens: 2.02 -> 0.63 ms with
// everything between queries and results (latent form before); one of
// 8192 13.1 -> 3.80 ms, four of 2048 4.48 -> 1.36 ms (with mla_prompt_kernel
// one step after the other; as it is it takes 7 % less).

#include <torch/all.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"

namespace vllm_amd {

namespace mla_prompt {

constexpr int LORA = 512;
constexpr int ROPE = 64;
constexpr int DK = LORA + ROPE;   // a latent row
constexpr int D = 128;            // a head's keys (without rotary), values
constexpr float NEG = -3.0e38f;
constexpr float GROWTH = 8.f;

// Exchanges of 16 B chunks / 32 B segments that keep LDS reads of 16 rows
// (plain fragments) and of 4 rows (transposing reads) off each other's
// banks, for rows of 128 and 256 B.
DEVINL int chunk128(int row, int c) { return c ^ ((row >> 1) & 7); }
DEVINL int chunk256(int row, int c) { return c ^ (row & 15); }
DEVINL int seg256(int row, int s) { return s ^ ((row & 3) << 1); }
DEVINL int seg256_chunk(int row, int c) {
  return seg256(row, c >> 1) * 2 + (c & 1);
}

// The powers of two that a block of keys and a row of queries are divided
// by on the way to fp16 (infinities and NaN by none). A row's is free, so
// its largest always lies below 2^14, with 2^28 of full precision under it.
DEVINL int exponent(float largest) {
  return (int)(__float_as_uint(largest) >> 23) - 127;
}
DEVINL int key_shift(float largest) {
  const int e = exponent(largest);
  return e == 128 || (e >= -2 && e <= 14) ? 0 : max(e, -60);
}
DEVINL int query_shift(float largest) {
  const int e = exponent(largest);
  return e == 128 ? 0 : max(e - 13, -60);
}
// exps of a head and request: two per 64 tokens.
DEVINL int exps_per_request(int S) { return (S + 63) / 64 * 2; }

// --------------------------------------------------------------------------
// Keys and values of EX_M context tokens for one head. Eight waves of
// 64 tokens x 64 columns, the first half of the columns keys, the second
// values. The latent is taken in steps of 64 through LDS, three stages,
// filled straight from global memory. The products are formed transposed
// (weights are the A operand; W_UV's fragments are transposing reads), so a
// lane ends up with runs of columns of one token. A workgroup goes on to
// the next heads without draining its stages (4 of them: 3 % of a prompt's
// time); the loop is one of two, for keys and for values, without a branch
// among its reads. Groups of heads are neighbours in the grid: an XCD meets
// every eighth group, whose weights stay in its L2. 3901 tokens x 128 heads:
// 0.19 ms, 690 TFLOP/s, 1.3 TB/s written.
constexpr int EX_M = 128;
constexpr int EX_K = 64;
constexpr int EX_THREADS = 8 * WAVE_SIZE;
constexpr int EX_STAGES = 3;
constexpr int EX_PART = EX_M * EX_K * 2;     // 16 KB: tokens, W_UK or W_UV
constexpr int EX_STAGE = 3 * EX_PART;
constexpr int EX_FILLS = EX_PART / 1024 / 8; // of each part, per wave
static_assert(EX_M == D && EX_PART == EX_K * D * 2);

template <typename Tag>
__launch_bounds__(EX_THREADS, 2) __global__
void mla_expand_kernel(short* __restrict__ k_out,   // [heads, reqs, S, D] fp16
                       short* __restrict__ v_out,   // [heads, reqs, S, D]
                       int* __restrict__ k_exp,     // [heads, reqs, S/64, 2]
                       short* __restrict__ pe_out,  // [reqs, S, ROPE]
                       const short* __restrict__ w_uk,  // [heads, D, LORA]
                       const short* __restrict__ w_uv,  // [heads, LORA, D]
                       const short* __restrict__ kv,    // [NB, BS, DK]
                       const int* __restrict__ block_table, int bt_stride,
                       const int* __restrict__ seq_lens, int block_size,
                       int num_decodes, int S, int heads, int per,
                       int write_pe) {
  const int h = blockIdx.x * per;
  const int t0 = blockIdx.y * EX_M;
  const int r = blockIdx.z;
  const int ctx = min(seq_lens[num_decodes + r], S);
  if (t0 >= ctx) return;
  __shared__ __align__(16) char lds[EX_STAGES * EX_STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l32 = lane & 31;
  const int half = lane >> 5;
  const int* bt = block_table + (int64_t)(num_decodes + r) * bt_stride;
  auto token = [&](int i) {   // its latent row; past the end the last one
    const int t = min(t0 + i, ctx - 1);
    const int b = t / block_size;
    return kv + ((int64_t)bt[b] * block_size + (t - b * block_size)) * DK;
  };

  // Each fill moves 8 rows of 128 B (tokens, W_UK) or 4 of 256 B (W_UV).
  const int frow = lane >> 3, fchunk = lane & 7;
  const short* src[3][EX_FILLS];
#pragma unroll
  for (int i = 0; i < EX_FILLS; ++i) {
    const int row = (wave * EX_FILLS + i) * 8 + frow;
    src[0][i] = token(row) + chunk128(row, fchunk) * 8;
    src[1][i] = w_uk + ((int64_t)h * D + row) * LORA +
                chunk128(row, fchunk) * 8;
    const int l = (wave * EX_FILLS + i) * 4 + (lane >> 4);
    src[2][i] = w_uv + ((int64_t)h * LORA + l) * D +
                seg256_chunk(l, lane & 15) * 8;
  }
  constexpr int STEPS = LORA / EX_K;
  const int all = min(per, heads - h) * STEPS;
  auto fill = [&](int s) {
    char* dst = lds + s % EX_STAGES * EX_STAGE + wave * EX_FILLS * 1024;
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int i = 0; i < EX_FILLS; ++i)
        lds_fill16(src[p][i] + (p == 2 ? s * (EX_K * D)
                                       : s % STEPS * EX_K +
                                             (p == 1 ? s / STEPS * D * LORA
                                                     : 0)),
                   dst + p * EX_PART + i * 1024);
  };

  const int wm = wave >> 2;          // 64 tokens
  const int wn = wave & 1;           // 64 columns ...
  const bool values = wave & 2;      // ... of the keys or of the values
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int reqs = gridDim.z;
  short* out = (values ? v_out : k_out) +
               (((int64_t)h * reqs + r) * S + t0) * D + wn * 64 + half * 8;
  fill(0);
  fill(1);
  auto run = [&](auto kind) {   // (no branch among the reads)
    constexpr bool VALUES = decltype(kind)::value;
#pragma unroll 1
    for (int s = 0; s < all; ++s) {
      // This stage has landed when only the next one's fills are under way;
      // past the barrier every wave is done with the stage before it.
      if (s + 1 < all) lds_fill_wait<3 * EX_FILLS>();
      else lds_fill_wait();
      lds_barrier();
      if (s + 2 < all) fill(s + 2);
      const char* t = lds + s % EX_STAGES * EX_STAGE;
#pragma unroll
      for (int kk = 0; kk < EX_K / 16; ++kk) {
        s16x8 x[2], w[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int row = wm * 64 + j * 32 + l32;
          x[j] = *reinterpret_cast<const s16x8*>(
              t + row * 128 + chunk128(row, kk * 2 + half) * 16);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if constexpr (VALUES) {
            const int l = kk * 16 + half * 8 + ((lane & 15) >> 2);
            const int seg = wn * 4 + i * 2 + ((lane >> 4) & 1);
            const char* at = t + 2 * EX_PART + (lane & 3) * 8;
            const s16x4 a = lds_read_tr(at + l * 256 + seg256(l, seg) * 32);
            const s16x4 b =
                lds_read_tr(at + (l + 4) * 256 + seg256(l + 4, seg) * 32);
            w[i] = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
          } else {
            const int row = wn * 64 + i * 32 + l32;
            w[i] = *reinterpret_cast<const s16x8*>(
                t + EX_PART + row * 128 + chunk128(row, kk * 2 + half) * 16);
          }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = mfma32<Tag>(w[i], x[j], acc[i][j]);
      }
      reads_ahead<VALUES ? 9 : 6, VALUES ? 3 : 2, EX_K / 16 * 2, 2>();
      if ((s + 1) % STEPS) continue;
      if constexpr (!VALUES) {
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
              mx = __builtin_amdgcn_fmed3f(mx, fabsf(acc[i][j][e]), INFINITY);
        int shift = 0;
        if (__any(!(mx < 32768.f)) || !__any(mx >= 0.25f)) {
          shift = key_shift(__uint_as_float(__builtin_amdgcn_readfirstlane(
              __float_as_uint(wave_reduce_max(mx)))));
          const float f = __builtin_ldexpf(1.f, -shift);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] *= f;
        }
        if (lane == 0 && t0 + wm * 64 < ctx)
          k_exp[((int64_t)(h + s / STEPS) * reqs + r) * exps_per_request(S) +
                (t0 / 64 + wm) * 2 + wn] = shift;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = wm * 64 + j * 32 + l32;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int b = 0; b < 4; b += 2) {
            f32x16& c = acc[i][j];
            const i32x4 w = VALUES ? row_chunk<Tag>(c, b)
                                   : row_chunk<FP16Tag>(c, b);
            if (t0 + row < ctx)
              *reinterpret_cast<i32x4*>(out + row * D + i * 32 + b * 8) = w;
#pragma unroll
            for (int e = 0; e < 8; ++e) c[b * 4 + e] = 0.f;
          }
      }
      out += (int64_t)reqs * S * D;
    }
  };
  if (values) run(std::true_type{});
  else run(std::false_type{});
  if (write_pe && h == 0) {
    for (int c = threadIdx.x; c < EX_M * 8; c += EX_THREADS)
      if (t0 + (c >> 3) < ctx)
        *reinterpret_cast<i32x4*>(
            pe_out + ((int64_t)r * S + t0 + (c >> 3)) * ROPE + (c & 7) * 8) =
            *reinterpret_cast<const i32x4*>(token(c >> 3) + LORA +
                                            (c & 7) * 8);
  }
}

// --------------------------------------------------------------------------
// Causal attention, 128 tokens of one head a workgroup, four waves of 32
// tokens, 64 keys a tile: 32x32x16 products S^T = K Q^T (a lane holds 32
// keys of one token) and O^T = V^T P^T with V^T by transposing reads, as
// for ordinary heads; per tile 24 + 32 products a wave (weights are hi + lo),
// 40 KB of fragment reads and 32 exponentials a lane, so the matrix cores
// bound it. As there (attention_prefill.h), a tile's maximum and weights are
// taken between the products of the next tile's scores and of its own results;
// two places of keys and of values, filled straight from global memory, one
// barrier a tile: 80 KB, two workgroups a CU. Accumulators are rescaled when a
// maximum has grown by 2^8. 3901 tokens as above: 0.45 ms, 910 TFLOP/s with
// both halves of the weights (scores, weights and results one after the other
// 0.485). All tiles of a head run on one XCD, late ones (most keys) first;
// where fewer than eight heads run at a time, a head's tiles go to several.
constexpr int PA_M = 128;
constexpr int PA_KEYS = 64;
constexpr int PA_THREADS = 4 * WAVE_SIZE;
constexpr int PA_K = PA_KEYS * D * 2;          // bytes: keys, values
constexpr int PA_PE = PA_KEYS * ROPE * 2;      // rotary parts
constexpr int PA_KEY_BYTES = PA_K + PA_PE;     // two places, then two of values

DEVINL float half_max(float x) {
  const auto sw = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  const unsigned lo = sw[0], hi = sw[1];
  return fmaxf(__uint_as_float(lo), __uint_as_float(hi));
}

template <typename Tag>
__launch_bounds__(PA_THREADS, 2) __global__
void mla_prompt_kernel(short* __restrict__ out,            // [T, Hq, D]
                       const short* __restrict__ q_nope,   // [T, Hq, D]
                       int64_t q_row, int64_t q_head,      // its strides
                       const short* __restrict__ q_pe,     // [T, Hq, ROPE]
                       const short* __restrict__ k,        // [heads, reqs, S, D]
                       const short* __restrict__ v,
                       const int* __restrict__ k_exp,
                       const short* __restrict__ pe,       // [reqs, S, ROPE]
                       const int* __restrict__ query_start_loc,
                       const int* __restrict__ seq_lens, float scale_log2,
                       int num_heads, int head0, int heads, int num_decodes,
                       int S, int tiles) {
  const int lanes = min(heads, 8);
  const int seq = (int)blockIdx.x / lanes;
  const int h = seq / tiles * lanes + (int)blockIdx.x % lanes;
  if (h >= heads) return;
  const int r = blockIdx.y;
  const int req = num_decodes + r;
  const int q_start = query_start_loc[req];
  const int ql = query_start_loc[req + 1] - q_start;
  const int tile = (ql + PA_M - 1) / PA_M - 1 - seq % tiles;
  const int ctx = min(seq_lens[req], S);
  if (tile < 0 || ctx < ql) return;
  const int pos0 = ctx - ql;             // of the portion's first token
  const int row0 = tile * PA_M;

  __shared__ __align__(16) char lds[2 * (PA_KEY_BYTES + PA_K)];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l32 = lane & 31;
  const int half = lane >> 5;
  const int tok = row0 + wave * 32 + l32;
  const int tok_safe = min(tok, ql - 1);
  const int qpos = pos0 + tok_safe;

  const int kt_end = (pos0 + min(row0 + PA_M, ql) - 1) / PA_KEYS + 1;
  const int* ke =
      k_exp + ((int64_t)h * gridDim.y + r) * exps_per_request(S);
  int shifted = 0;
  for (int i = lane; i < kt_end * 2; i += WAVE_SIZE) shifted |= ke[i];

  s16x8 qf[(D + ROPE) / 16];
  {
    const short* qn = q_nope + (q_start + tok_safe) * q_row +
                      (head0 + h) * q_head + half * 8;
    const short* qp = q_pe + ((int64_t)(q_start + tok_safe) * num_heads +
                              head0 + h) * ROPE + half * 8;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
      qf[kk] = *reinterpret_cast<const s16x8*>(qn + kk * 16);
#pragma unroll
    for (int kk = 0; kk < ROPE / 16; ++kk)
      qf[D / 16 + kk] = *reinterpret_cast<const s16x8*>(qp + kk * 16);
  }
  // A bf16 query has fewer bits than fp16; the scale takes its power of two
  // back.
  float scale = scale_log2;
  if constexpr (std::is_same_v<Tag, BF16Tag>) {
    float mx = 0.f;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        mx = fmaxf(mx, fabsf(bf16_to_f32(qf[kk][e])));
    const int shift = query_shift(half_max(mx));
    const float f = __builtin_ldexpf(1.f, -shift);
    scale = __builtin_ldexpf(scale_log2, shift);
#pragma unroll
    for (int kk = 0; kk < (D + ROPE) / 16; ++kk) {
      i32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = bf16_to_f32(qf[kk][e * 2]) * f;
        const float b = bf16_to_f32(qf[kk][e * 2 + 1]) * f;
        w[e] = kk < D / 16 ? pack2<FP16Tag>(a, b) : pack2<BF16Tag>(a, b);
      }
      qf[kk] = __builtin_bit_cast(s16x8, w);
    }
  }

  const int64_t base = ((int64_t)h * gridDim.y + r) * S;
  const short* kb = k + base * D;
  const short* vb = v + base * D;
  const short* pb = pe + (int64_t)r * S * ROPE;
  // Rows past the context repeat the last one: their weight is zero, and
  // what was never written could be NaN.
  auto fill_keys = [&](int kt, int place) {
    char* dst = lds + place * PA_KEY_BYTES;
    const int last = ctx - 1 - kt * PA_KEYS;
    const int64_t t0 = (int64_t)kt * PA_KEYS;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (wave * 4 + i) * 4 + (lane >> 4);
      lds_fill16(kb + t0 * D,
                 (uint32_t)(min(row, last) * D + chunk256(row, lane & 15) * 8) *
                     2,
                 dst + (wave * 4 + i) * 1024);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = (wave * 2 + i) * 8 + (lane >> 3);
      lds_fill16(pb + t0 * ROPE,
                 (uint32_t)(min(row, last) * ROPE +
                            chunk128(row, lane & 7) * 8) * 2,
                 dst + PA_K + (wave * 2 + i) * 1024);
    }
  };
  auto fill_values = [&](int kt, int place) {
    char* dst = lds + 2 * PA_KEY_BYTES + place * PA_K;
    const int last = ctx - 1 - kt * PA_KEYS;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (wave * 4 + i) * 4 + (lane >> 4);
      lds_fill16(vb + (int64_t)kt * PA_KEYS * D,
                 (uint32_t)(min(row, last) * D +
                            seg256_chunk(row, lane & 15) * 8) * 2,
                 dst + (wave * 4 + i) * 1024);
    }
  };

  float m_run = NEG, l_run = 0.f;   // log2 domain; l: the keys of this lane
  f32x16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[i][e] = 0.f;

  const int wave_first = pos0 + row0 + wave * 32;
  const int wave_last = pos0 + min(row0 + wave * 32 + 31, ql - 1);

  // Fragments of a step in the order of their products: the first and the
  // second 32 keys of the next tile's scores (one product each), then the four
  // chunks of 16 keys of this one's results (two, by the weights' parts).
  constexpr int KF = (D + ROPE) / 16, DS = D / 32;
  constexpr int QK = 2 * KF, ALL = QK + 4 * DS;
  int k_at[KF], v_at[DS];    // first fragments of a tile, in its bytes
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk)
    k_at[kk] = l32 * 256 + chunk256(l32, kk * 2 + half) * 16;
#pragma unroll
  for (int kk = 0; kk < ROPE / 16; ++kk)
    k_at[D / 16 + kk] = PA_K + l32 * 128 + chunk128(l32, kk * 2 + half) * 16;
#pragma unroll
  for (int i = 0; i < DS; ++i) {
    const int row = half * 4 + ((lane & 15) >> 2);
    v_at[i] = row * 256 + seg256(row, i * 2 + ((lane >> 4) & 1)) * 32 +
              (lane & 3) * 8;
  }
  auto fragment = [&](int m, int k_place, int v_place, auto again) -> s16x8 {
    if (m < QK) {   // (the moves of rows 16 and 32 apart are the same)
      int at = k_at[m % KF];
      if constexpr (decltype(again)::value) {
        // Formed anew, not kept: there is no register left for it.
        int l = lane;
        asm volatile("" : "+v"(l));
        const int row = l & 31, c = m % KF * 2 + (l >> 5);
        at = m % KF < D / 16
                 ? row * 256 + chunk256(row, c) * 16
                 : PA_K + row * 128 + chunk128(row, c - D / 8) * 16;
      }
      return *reinterpret_cast<const s16x8*>(
          lds + k_place * PA_KEY_BYTES +
          m / KF * 32 * (m % KF < D / 16 ? 256 : 128) + at);
    }
    const char* at = lds + 2 * PA_KEY_BYTES + v_place * PA_K +
                     (m - QK) / DS * 16 * 256 + v_at[(m - QK) % DS];
    const s16x4 a = lds_read_tr(at), b = lds_read_tr(at + 8 * 256);
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  const f32x16 zero = {};

  auto run = [&](auto shifts) {
    constexpr bool SHIFTS = decltype(shifts)::value;
    // Fragments read ahead. (Scratch for the rare form with shifts would cost
    // all launches: one prompt of 22 tokens 6.9 us with 44 B of it, 6.6 with
    // none.)
    constexpr int AHEAD = SHIFTS ? 1 : 4;
    // Product m of the scores t of tile kt.
    auto score = [&](const int kt, const int m, const s16x8 f,
                     f32x16 (&t)[2]) {
      const int n = m / KF, kk = m % KF;
      if (kk < D / 16)
        t[n] = mfma32<FP16Tag>(f, qf[kk], kk == 0 ? zero : t[n]);
      else
        t[n] = mfma32<Tag>(f, qf[kk], t[n]);
      if constexpr (SHIFTS) {
        if (kk == D / 32 - 1)
          t[n] *= __builtin_ldexpf(1.f, min(ke[kt * 2] - ke[kt * 2 + 1], 127));
        if (kk == D / 16 - 1) t[n] *= __builtin_ldexpf(1.f, ke[kt * 2 + 1]);
      }
    };
    // One tile: its scores s become weights and results, between the products
    // of the next one's scores t (MORE; where there is none, of what lies
    // there).
    auto tile_step = [&](const int kt, f32x16 (&s)[2], f32x16 (&t)[2],
                         const int place, auto more) {
      constexpr bool MORE = decltype(more)::value;
      constexpr int FIRST = MORE ? 0 : QK;
      if constexpr (MORE) {
        // (Of either place the last read lies before the barrier.)
        if (kt + 1 < kt_end) fill_values(kt + 1, 1 - place);
        if (kt + 2 < kt_end) fill_keys(kt + 2, place);
      }
      if (kt * PA_KEYS <= wave_last) {   // else no key for these tokens
        s16x8 frag[AHEAD], p_hi[4], p_lo[4];
        const int nt = min(kt + 1, kt_end - 1);
        auto read = [&](int m) {
          if (m >= FIRST && m < ALL)
            frag[m % AHEAD] = fragment(m, 1 - place, place, shifts);
        };
        auto product = [&](int m) {
          const s16x8 f = frag[m % AHEAD];
          if (m < QK) {
            score(nt, m, f, t);
          } else {
            const int c = (m - QK) / DS, i = (m - QK) % DS;
            o[i] = mfma32<Tag>(f, p_lo[c], o[i]);
            o[i] = mfma32<Tag>(f, p_hi[c], o[i]);
          }
          read(m + AHEAD);
        };
        // Register e of s[n] is key n*32 + 8*(e/4) + 4*half + e%4.
        if (kt * PA_KEYS + PA_KEYS - 1 > wave_first) {
          const int left = qpos - kt * PA_KEYS - half * 4;
#pragma unroll
          for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e)
              s[n][e] = n * 32 + 8 * (e >> 2) + (e & 3) <= left ? s[n][e] : NEG;
        }
#pragma unroll
        for (int m = FIRST; m < FIRST + AHEAD; ++m) read(m);
        float mx = NEG;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int e = g * 4; e < g * 4 + 4; ++e) {
            mx = __builtin_amdgcn_fmed3f(mx, s[0][e], INFINITY);
            mx = __builtin_amdgcn_fmed3f(mx, s[1][e], INFINITY);
          }
          if constexpr (MORE) {
#pragma unroll
            for (int m = KF * g / 4; m < KF * (g + 1) / 4; ++m) product(m);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        mx = half_max(mx) * scale;
        if (__any(mx - m_run > GROWTH)) {
          const float m_new = fmaxf(m_run, mx);
          const float f = __builtin_amdgcn_exp2f(m_run - m_new);
          l_run *= f;
#pragma unroll
          for (int i = 0; i < DS; ++i) o[i] *= f;
          m_run = m_new;
        }
        // --- weights, and O^T += V^T P^T, 16 keys at a time ----------------
        // Half a chunk of weights a group, then as many products as weights
        // are there for.
        constexpr int TO[9] = {KF, 16, 20, 25, 28, 30, 32, 34, 36};
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          __builtin_amdgcn_sched_barrier(0);
          const int c = g / 2;
          i32x4 hi = {}, lo = {};
          if (g % 2) {
            hi = __builtin_bit_cast(i32x4, p_hi[c]);
            lo = __builtin_bit_cast(i32x4, p_lo[c]);
          }
#pragma unroll
          for (int j = g % 2 * 2; j < g % 2 * 2 + 2; ++j) {
            const int e = (c & 1) * 8 + j * 2;
            const float p0 = __builtin_amdgcn_exp2f(
                __builtin_fmaf(s[c >> 1][e], scale, -m_run));
            const float p1 = __builtin_amdgcn_exp2f(
                __builtin_fmaf(s[c >> 1][e + 1], scale, -m_run));
            hi[j] = pack2<Tag>(p0, p1);
            l_run += p0 + p1;
            lo[j] = pack2<Tag>(p0 - unpack_lo<Tag>(hi[j]),
                               p1 - unpack_hi<Tag>(hi[j]));
          }
          p_hi[c] = __builtin_bit_cast(s16x8, hi);
          p_lo[c] = __builtin_bit_cast(s16x8, lo);
#pragma unroll
          for (int m = TO[g]; m < TO[g + 1]; ++m)
            if (m >= FIRST) product(m);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = TO[8]; m < ALL; ++m) product(m);
      }
      if constexpr (MORE) lds_fill_wait();
      lds_barrier();
    };

    fill_keys(0, 0);
    fill_values(0, 0);
    if (kt_end > 1) fill_keys(1, 1);
    lds_fill_wait();
    lds_barrier();
    f32x16 sa[2], sb[2];
#pragma unroll
    for (int m = 0; m < QK; ++m) {
      score(0, m, fragment(m, 0, 0, shifts), sa);
      if (SHIFTS && m % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if (kt_end > 1) lds_barrier();   // the first keys' place is free
    int kt = 0;
#pragma unroll 1
    for (; kt + 1 < kt_end; kt += 2) {
      tile_step(kt, sa, sb, 0, std::true_type{});
      tile_step(kt + 1, sb, sa, 1, std::true_type{});
    }
    if (kt < kt_end) tile_step(kt, sa, sb, 0, std::false_type{});
  };
  if (__any(shifted != 0)) run(std::true_type{});
  else run(std::false_type{});

  l_run += __shfl_xor(l_run, 32, 64);
  const float inv_l = 1.f / l_run;
  short* ob = out + ((int64_t)(q_start + tok) * num_heads + head0 + h) * D +
              half * 8;
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    o[i] *= inv_l;
#pragma unroll
    for (int b = 0; b < 4; b += 2) {
      const i32x4 w = row_chunk<Tag>(o[i], b);
      if (tok < ql) *reinterpret_cast<i32x4*>(ob + i * 32 + b * 8) = w;
    }
  }
}

}  // namespace mla_prompt

// Prompt portions (requests num_decodes..) of a step; out, q_nope and q_pe
// [T, Hq, 128 / 128 / 64] cover the whole step. scratch holds per head
// 2 x [reqs, S, 128] and once [reqs, S, 64] values, S >= every context; as
// many heads as fit run at a time. exps [heads at a time, reqs,
// ceil(S / 64), 2] are the keys' exponents.
void mla_prompt_attention(torch::Tensor out, torch::Tensor q_nope,
                          torch::Tensor q_pe, torch::Tensor w_uk,
                          torch::Tensor w_uv, torch::Tensor kv_cache,
                          torch::Tensor block_table,
                          torch::Tensor query_start_loc,
                          torch::Tensor seq_lens, double scale,
                          int64_t num_decodes, int64_t max_query_len,
                          int64_t S, torch::Tensor scratch,
                          torch::Tensor exps) {
  using namespace mla_prompt;
  TORCH_CHECK(q_nope.dim() == 3 && q_nope.size(2) == D &&
              q_pe.dim() == 3 && q_pe.size(2) == ROPE &&
              kv_cache.dim() == 3 && kv_cache.size(2) == DK,
              "mla prompts: heads of 128 + 64 over a latent of 512 + 64");
  const int64_t T = q_nope.size(0), Hq = q_nope.size(1);
  TORCH_CHECK(w_uk.dim() == 3 && w_uk.size(0) == Hq && w_uk.size(1) == D &&
              w_uk.size(2) == LORA && w_uv.dim() == 3 &&
              w_uv.size(0) == Hq && w_uv.size(1) == LORA &&
              w_uv.size(2) == D);
  TORCH_CHECK(out.dim() == 3 && out.size(0) == T && out.size(1) == Hq &&
              out.size(2) == D && q_pe.size(0) == T && q_pe.size(1) == Hq);
  TORCH_CHECK(out.is_contiguous() && q_pe.is_contiguous() &&
              w_uk.is_contiguous() && w_uv.is_contiguous() &&
              kv_cache.is_contiguous() && scratch.is_contiguous());
  TORCH_CHECK(q_nope.stride(2) == 1 && q_nope.stride(0) % 8 == 0 &&
              q_nope.stride(1) % 8 == 0);
  for (const auto& x : {q_nope, w_uk, w_uv, kv_cache, scratch})
    TORCH_CHECK((uintptr_t)x.data_ptr() % 16 == 0);
  const auto type = q_nope.scalar_type();
  TORCH_CHECK(type == torch::kBFloat16 || type == torch::kHalf);
  for (const auto& x : {out, q_pe, w_uk, w_uv, kv_cache, scratch})
    TORCH_CHECK(x.scalar_type() == type);
  const int64_t reqs = seq_lens.size(0) - num_decodes;
  if (reqs <= 0 || T <= num_decodes) return;
  TORCH_CHECK(query_start_loc.numel() > seq_lens.size(0));
  TORCH_CHECK(scale > 0 && S > 0 && max_query_len > 0 && reqs < 65536);
  const int64_t pe_size = reqs * S * ROPE, head_size = reqs * S * D;
  const int at_once = (int)std::min<int64_t>(
      Hq, (scratch.numel() - pe_size) / (2 * head_size));
  TORCH_CHECK(at_once >= 1, "mla prompts: scratch holds no head");
  TORCH_CHECK(exps.scalar_type() == torch::kInt32 && exps.is_contiguous() &&
              exps.numel() >= at_once * reqs * ((S + 63) / 64 * 2));
  short* pe = (short*)scratch.data_ptr();
  short* k = pe + pe_size;
  short* v = k + at_once * head_size;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const int tiles = ceil_div((int)std::min(max_query_len, S), PA_M);
  const int token_tiles = ceil_div((int)S, EX_M);
  auto launch = [&](auto tag) {
    using Tag = decltype(tag);
    for (int h0 = 0; h0 < Hq; h0 += at_once) {
      const int heads = (int)std::min<int64_t>(at_once, Hq - h0);
      const int per = ceil_div(heads, 4) * token_tiles * reqs >= 256 ? 4 : 1;
      hipLaunchKernelGGL(
          (mla_expand_kernel<Tag>),
          dim3(ceil_div(heads, per), token_tiles, (int)reqs),
          dim3(EX_THREADS), 0,
          stream, k, v, exps.data_ptr<int>(), pe,
          (const short*)w_uk.data_ptr() + h0 * D * LORA,
          (const short*)w_uv.data_ptr() + h0 * D * LORA,
          (const short*)kv_cache.data_ptr(), block_table.data_ptr<int>(),
          (int)block_table.size(1), seq_lens.data_ptr<int>(),
          (int)kv_cache.size(1), (int)num_decodes, (int)S, heads, per, h0 == 0);
      HIP_CHECK_KERNEL();
      const int lanes = std::min(heads, 8);
      hipLaunchKernelGGL(
          (mla_prompt_kernel<Tag>),
          dim3(ceil_div(heads, lanes) * lanes * tiles, (int)reqs),
          dim3(PA_THREADS),
          0, stream, (short*)out.data_ptr(), (const short*)q_nope.data_ptr(),
          q_nope.stride(0), q_nope.stride(1), (const short*)q_pe.data_ptr(),
          k, v, exps.data_ptr<int>(), pe, query_start_loc.data_ptr<int>(),
          seq_lens.data_ptr<int>(), (float)scale * 1.4426950408889634f,
          (int)Hq, h0, heads, (int)num_decodes, (int)S, tiles);
      HIP_CHECK_KERNEL();
    }
  };
  if (type == torch::kBFloat16) launch(BF16Tag{});
  else launch(FP16Tag{});
}

}  // namespace vllm_amd
