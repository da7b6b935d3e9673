// Product of a few rows with a tile of weight rows, weights streamed from HBM
// (gfx950): stream_linear.hip, moe.hip. Why it is laid out like this and what
// that gives: stream_linear.hip.
#pragma once

#include "common.h"

namespace vllm_amd {

constexpr int SP_K = 64;         // columns of K per step of a wave: 128 B
constexpr int SP_FILL = 1024;    // bytes of a fill: 8 rows x 128 B

// Places of a lane's pieces: 16 B chunk c of row r lies at c ^ (r / 2 & 7),
// so that the 16 rows of a fragment read meet no bank twice.
DEVINL uint32_t sp_place(uint32_t src_row, int row, int K) {
  return src_row * (uint32_t)(K * 2) +
         (((threadIdx.x & 7) ^ ((row >> 1) & 7)) * 16);
}

// LDS that a wave's gains take, of `steps` steps of K over `waves` waves.
constexpr __host__ __device__ int sp_gain_bytes(int steps, int waves) {
  return ((steps + waves - 1) / waves + 7) / 8 * SP_FILL;
}

struct Nothing {
  DEVINL void operator()() const {}
};

// NI: 16-row groups of weights; XG: groups of 8 rows of x; WV: waves that
// multiply (of NW in the workgroup), each with a ring of D steps.
// NORM: the rows of x are multiplied by gains, one for each column of K, on
// their way to the product, and their squares are summed beside it.
template <typename Tag, int NI, int XG, int WV, int D, bool NORM = false>
struct StreamProduct {
  static constexpr int MT = (XG + 1) / 2;      // 16-row groups of x
  static constexpr int FILLS = 2 * NI + XG;
  static constexpr int STEP = FILLS * SP_FILL;
  static constexpr int T = NI * MT;            // 16 x 16 tiles of sums
  static constexpr int RING = WV * D * STEP;
  static constexpr int TN = T + (NORM ? 1 : 0);   // and the squares
  static constexpr int SUMS = WV * TN * WAVE_SIZE * 16;
  static constexpr int LDS = RING > SUMS ? RING : SUMS;
  static_assert(!NORM || MT <= 4, "squares of 16 rows in each of four places");
  static_assert(D > 1 && (D - 1) * FILLS < 64, "what a wait can count");

  // Steps s0 .. s1 - 1 of K, every WV-th for this wave, beginning at the
  // `turn`-th of them. wat, xat: byte places in w and x of this lane's piece
  // of the i-th 8 rows. Afterwards sum(t) of every tile t of the workgroup;
  // tile i * MT + j is 16 weight rows by 16 rows of x: a lane holds weight
  // rows l4 * 4 .. + 3 of row l16. NORM: sum(T)[j] is the sum of squares of
  // row l16 of the j-th 16 over these steps; the gains take
  // sp_gain_bytes(s1 - s0, WV) of LDS behind LDS for each wave.
  // early(): what the caller loads for the end, asked for behind the first
  // fills, which it would keep waiting before them.
  template <typename Early = Nothing>
  static DEVINL void run(char* lds, const int wave, const int s0,
                         const int s1, const int turn_seed,
                         const char* __restrict__ w,
                         const uint32_t (&wat)[2 * NI],
                         const char* __restrict__ x,
                         const uint32_t (&xat)[XG],
                         const char* __restrict__ gains = nullptr,
                         const Early& early = Early{}) {
    const int lane = threadIdx.x % WAVE_SIZE;
    const int l16 = lane & 15;
    const int l4 = lane >> 4;
    const int n =
        wave < WV && s1 - s0 > wave ? (s1 - s0 - wave + WV - 1) / WV : 0;
    const int turn = n > 0 ? (int)((unsigned)turn_seed % (unsigned)n) : 0;
    char* ring = lds + wave * (D * STEP);
    // All of this wave's gains, 128 B a step in the order of the steps, before
    // anything else: the first wait for a step is one for them too.
    char* gain = lds + LDS + wave * sp_gain_bytes(s1 - s0, WV);
    if constexpr (NORM) {
      for (int q = 0; q * 8 < n; ++q)
        lds_fill16(gains,
                   (uint32_t)(s0 + wave +
                              min(q * 8 + (lane >> 3), n - 1) * WV) *
                           (SP_K * 2) +
                       (lane & 7) * 16,
                   gain + q * SP_FILL);
    }
    auto fill = [&](int i, int slot) {
      i = min(i, n - 1) + turn;
      const int64_t k = (int64_t)(s0 + wave + (i >= n ? i - n : i) * WV) *
                        (SP_K * 2);
      char* to = ring + slot * STEP;
#pragma unroll
      for (int j = 0; j < 2 * NI; ++j)
        lds_fill16_once(w + k, wat[j], to + j * SP_FILL);
#pragma unroll
      for (int j = 0; j < XG; ++j)
        lds_fill16(x + k, xat[j], to + (2 * NI + j) * SP_FILL);
    };

    f32x4 acc[NI][MT];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The product is formed transposed. (Of 8 rows the upper lanes repeat
    // the lower.)
    const int xrow = XG == 1 ? l16 & 7 : l16;
    // Rows by themselves: their sums of squares are the diagonal. (Matrix cores
    // have time; by the vector ALU, in a chain, the same within 2 %.)
    f32x4 squares[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) squares[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int slot, int i) {
      const char* from = ring + slot * STEP;
      s16x8 wf[2][NI], xf[2][MT];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
          wf[u][i] = *reinterpret_cast<const s16x8*>(
              from + (i * 16 + l16) * 128 +
              ((u * 4 + l4) ^ ((l16 >> 1) & 7)) * 16);
#pragma unroll
        for (int j = 0; j < MT; ++j)
          xf[u][j] = *reinterpret_cast<const s16x8*>(
              from + 2 * NI * SP_FILL + (j * 16 + xrow) * 128 +
              ((u * 4 + l4) ^ ((xrow >> 1) & 7)) * 16);
      }
      if constexpr (NORM) {
        i += turn;
        const char* g = gain + (i >= n ? i - n : i) * (SP_K * 2) + l4 * 16;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const i32x4 gf = *reinterpret_cast<const i32x4*>(g + u * 64);
#pragma unroll
          for (int j = 0; j < MT; ++j) {
            squares[j] = mfma16<Tag>(xf[u][j], xf[u][j], squares[j]);
            i32x4 f = __builtin_bit_cast(i32x4, xf[u][j]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              f[e] = pack2<Tag>(unpack_lo<Tag>(f[e]) * unpack_lo<Tag>(gf[e]),
                                unpack_hi<Tag>(f[e]) * unpack_hi<Tag>(gf[e]));
            xf[u][j] = __builtin_bit_cast(s16x8, f);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j)
            acc[i][j] = mfma16<Tag>(wf[u][i], xf[u][j], acc[i][j]);
    };
    if (n == 0) early();
    if (n > 0) {
      // Short waves fill the last step more than once: the counts that the
      // waits go by stay the same.
#pragma unroll
      for (int d = 0; d < D - 1; ++d) fill(d, d);
      early();
      int slot = 0, i = 0;
      for (; i + D - 1 < n; ++i) {
        fill(i + D - 1, slot == 0 ? D - 1 : slot - 1);
        lds_fill_wait<(D - 1) * FILLS>();
        asm volatile("" ::: "memory");
        multiply(slot, i);
        // Read before it is filled again.
        lds_wait();
        slot = slot + 1 == D ? 0 : slot + 1;
      }
      lds_fill_wait();
      asm volatile("" ::: "memory");
      for (; i < n; ++i) {
        multiply(slot, i);
        slot = slot + 1 == D ? 0 : slot + 1;
      }
    }
    f32x4* red = reinterpret_cast<f32x4*>(lds);
    __syncthreads();
    if (wave < WV) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          red[(wave * TN + i * MT + j) * WAVE_SIZE + lane] = acc[i][j];
      if constexpr (NORM) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          float own = squares[j][0];   // of row l16, in group l16 / 4
#pragma unroll
          for (int r = 1; r < 4; ++r)
            own = (l16 & 3) == r ? squares[j][r] : own;
          v[j] = __shfl(own, (l16 >> 2) * 16 + l16, WAVE_SIZE);
        }
        red[(wave * TN + T) * WAVE_SIZE + lane] = v;
      }
    }
    __syncthreads();
  }

  static DEVINL f32x4 sum(const char* lds, int t) {
    const f32x4* red = reinterpret_cast<const f32x4*>(lds) +
                       threadIdx.x % WAVE_SIZE;
    f32x4 v = red[t * WAVE_SIZE];
#pragma unroll
    for (int q = 1; q < WV; ++q) v += red[(q * TN + t) * WAVE_SIZE];
    return v;
  }
};

}  // namespace vllm_amd
