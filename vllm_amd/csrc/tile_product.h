// Product of a tile of rows with a tile of weight rows by four waves, one
// a SIMD (gfx950): acc += W[TN, K] @ X[TM, K]^T, 16-bit operands in
// LDS, fp32 sums in accumulation registers. Compile files that use it
// without -amdgpu-mfma-vgpr-form: 256 accumulators a lane leave no room in
// the vector registers.
//
// What bounds it. Large products the chip's power: the matrix cores are busy
// three quarters of the cycles, at 1.7 to 1.8 GHz. Products of 16 x 16 x 32
// move half the accumulators per flop that those of 32 x 32 x 16 do (random
// values from registers alone: 2.02 and 1.77 PFLOP/s). Small ones what a CU
// takes in: 46 to 60 GB/s of rows from L2 and weights from HBM together.
//  * A wave of 128 x 128 reads 16 fragments of 16 x 32 from LDS for 64 products
//    (half of what LDS gives; eight waves of 64 x 128 read 96 B a clock, and
//    with what is filled that is all there is). With one wave a SIMD nothing
//    else hides a wait, so nothing waits: fragments of the next 32 columns are
//    read between this step's products, the order of products being that in
//    which fragments arrive (pinned by scheduling barriers: the compiler would
//    move reads to their use);
//  * A wave issues an instruction every four cycles and a product takes 16, so
//    three others fit behind one. Reads and fills stand evenly between single
//    products, and a fill is one piece with its product, its place set before
//    it and its load behind it. Cycles a stage where all operands are in L2,
//    128 x 256 and 256 x 256: 1280 and 2310; with reads and fills of four
//    instructions between groups of four products 1480 and 2490 (8 experts of
//    4096 x 768, 4 each of 318 tokens 75.2 us, so 69.6; layers of K = 1024 to
//    2048 gain 2.6 %); products of 32 x 32 x 16, which hide more behind
//    each, 1230 and 2210.
//  * fills go straight from global memory to LDS: all at once they back up
//    behind each other;
//  * one barrier per 64 columns, before the last of their two steps, by
//    when all of their fragments are in registers. From there on their
//    places are filled again, that of the rows first. (Beside 256 x 256
//    tiles LDS has two places for rows and three for weights, which come
//    from further away.)
// 8192 x 4096 x 14336 in bf16: 1.50 PFLOP/s, 8192 x 28672 x 4096 1.43, 2048 x
// 8192 x 4096 1.40 (32 x 32 x 16 1.43, 1.36 and 1.29; eight waves by halves in
// turn 1.0; the tuned library 1.60 and 1.57 of the first two).
#pragma once

#include <type_traits>

#include "common.h"

namespace vllm_amd {

constexpr int TP_K = 64;                  // columns of a stage: 128 B lines
constexpr int TP_ROW = TP_K * 2;          // bytes of a row of a stage
constexpr int TP_FILL = 1024;             // bytes of a fill: 8 rows
constexpr int TP_THREADS = 4 * WAVE_SIZE;

// 16 B chunk c of row r of a stage lies at c ^ tp_swap(r), so that the rows
// of a fragment read meet no bank twice.
DEVINL int tp_swap(int row) { return (row >> 1) & 7; }

// Order of the fragments of a step (weights and rows in turn) and of its
// products: each as soon as both fragments are there.
template <int NI, int J> struct TpOrder {
  bool w[NI + J]{};
  int ix[NI + J]{}, i[NI * J + 1]{}, j[NI * J + 1]{};
  constexpr TpOrder() {
    int nw = 0, na = 0, n = 0;
    for (int r = 0; r < NI + J; ++r) {
      const bool tw = nw < NI && (nw <= na || na == J);
      w[r] = tw;
      ix[r] = tw ? nw : na;
      for (int q = 0; q < (tw ? na : nw); ++q) {
        i[n] = tw ? nw : q;
        j[n] = tw ? q : na;
        ++n;
      }
      (tw ? nw : na)++;
    }
  }
};

// What a lane of a fill reads: base + at, base the same in all lanes.
struct FillSource {
  const void* base;
  uint32_t at;
};

// WGM: waves along the rows (4 / WGM along the weights). NG, MG: 32-row
// groups of weights and of rows a wave takes. PA, PW: stages of rows and of
// weights that LDS holds. The waves' groups of rows alternate, so that in a
// tile with few rows they have as many each.
template <typename Tag, int WGM, int NG, int MG, int PA, int PW>
struct TileProduct {
  static constexpr int WGN = 4 / WGM;
  static constexpr int NI = NG * 2;          // 16-row groups of weights
  static constexpr int TM = WGM * MG * 32;
  static constexpr int TN = WGN * NG * 32;
  static constexpr int AB = TM * TP_ROW;     // bytes of a stage
  static constexpr int WB = TN * TP_ROW;
  static constexpr int FA = TM / 8 / 4;      // fills a wave
  static constexpr int FW = TN / 8 / 4;
  static constexpr int LDS = PA * AB + PW * WB;
  static constexpr int WW = NG * 32;         // weight rows of a wave
  static_assert(PA >= 2 && PW >= PA && LDS <= 160 * 1024);

  // First row in the tile of 16-row group j of a wave that is wm-th along
  // the rows.
  static DEVINL int row_of(int j, int wm) {
    return (j / 2 * WGM + wm) * 32 + j % 2 * 16;
  }

  // from_a(stage, i) and from_w: the sources of the wave's i-th fill of 8 rows
  // of a stage, rows (wave * FA + i) * 8 .. of the tile; ONCE: weights that
  // nobody else reads. done(J, acc) gets the sums of the J 16-row groups of
  // this wave in the 32-row groups that hold any of `rows`: register r of
  // acc[i][j] is weight row i*16 + 4*l4 + r of the wave, row l16 of its group
  // j.
  template <bool ONCE, typename FromA, typename FromW, typename Done>
  static DEVINL void run(char* lds, const int steps, const int rows,
                         FromA from_a, FromW from_w, Done done) {
    const int wave =
        __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
    const int wm = wave / WGN;
    const int groups = (min(rows, TM) + 31) / 32;
    const int mine = (groups - wm + WGM - 1) / WGM;
    auto go = [&](auto n) {
      constexpr int J = decltype(n)::value * 2;
      f32x4 acc[NI][J > 0 ? J : 1];
      loop<ONCE, J>(lds, steps, wave, from_a, from_w, acc);
      done(std::integral_constant<int, J>{}, acc);
    };
    if (mine >= MG) go(std::integral_constant<int, MG>{});
    else if (MG > 3 && mine == 3) go(std::integral_constant<int, 3>{});
    else if (MG > 2 && mine == 2) go(std::integral_constant<int, 2>{});
    else if (MG > 1 && mine == 1) go(std::integral_constant<int, 1>{});
    else go(std::integral_constant<int, 0>{});
  }

 private:
  // The fills of n whole stages may be under way (where rows and weights are
  // as far ahead; none elsewhere).
  template <int MAX> static DEVINL void wait_but(int n) {
    if constexpr (PA == PW && MAX > 0) {
      if (n >= MAX) return lds_fill_wait<MAX * (FA + FW)>();
      return wait_but<MAX - 1>(n);
    }
    lds_fill_wait();
  }

  // Reads of a step (F, evenly over the first SPAN quarters of its M products)
  // that come before product q.
  template <int M, int F, int SPAN> static constexpr int reads_by(int q) {
    const int n = (4 * F * q + M * SPAN - 1) / (M * SPAN);
    return n < F ? n : F;
  }

  template <bool ONCE, int J, typename FromA, typename FromW, int JA>
  static DEVINL void loop(char* lds, const int steps, const int wave,
                          FromA from_a, FromW from_w, f32x4 (&acc)[NI][JA]) {
    constexpr TpOrder<NI, J> O{};
    constexpr int M = NI * J, F = J > 0 ? NI + J : 0;
    static_assert(M == 0 || (M >= FA && M >= FW));
    const int lane = threadIdx.x % WAVE_SIZE;
    const int l16 = lane & 15;
    const int l4 = lane >> 4;
    const int wm = wave / WGN, wn = wave % WGN;
    int at[2];   // byte places of this lane's fragments of a group
#pragma unroll
    for (int k = 0; k < 2; ++k)
      at[k] = l16 * TP_ROW + ((k * 4 + l4) ^ tp_swap(l16)) * 16;
    char* const wlds = lds + PA * AB;
    const char* const w0 = wlds + wn * WW * TP_ROW;
    char* const a_to = lds + wave * FA * TP_FILL;    // this wave's fills
    char* const w_to = wlds + wave * FW * TP_FILL;
    auto fa = [&](int s, int i, int place) {
      const FillSource v = from_a(s, i);
      lds_fill16(v.base, v.at, a_to + place * AB + i * TP_FILL);
    };
    auto fw = [&](int s, int i, int place) {
      const FillSource v = from_w(s, i);
      char* const to = w_to + place * WB + i * TP_FILL;
      if constexpr (ONCE) lds_fill16_once(v.base, v.at, to);
      else lds_fill16(v.base, v.at, to);
    };
    s16x8 af[2][J > 0 ? J : 1], wf[2][NI];
    auto read = [&](int to, int ap, int wp, int k, auto nth) {
      constexpr int r = decltype(nth)::value, x = O.ix[r];
      if constexpr (O.w[r])
        wf[to][x] = *reinterpret_cast<const s16x8*>(
            w0 + wp * WB + x * 16 * TP_ROW + at[k]);
      else
        af[to][x] = *reinterpret_cast<const s16x8*>(
            lds + ap * AB + row_of(x, wm) * TP_ROW + at[k]);
    };
    // Products from fragments CUR; between them, evenly over the first SPAN
    // quarters, the reads of the next step's fragments, and n fills: in one
    // piece with a product where they are JOINED, else as the caller fills.
    auto step = [&](auto cur, auto span, auto reads, auto n, auto joined,
                    auto once, auto from, char* to, auto fill) {
      constexpr int CUR = decltype(cur)::value, N = decltype(n)::value;
      constexpr int SPAN = decltype(span)::value;
      if constexpr (M == 0) {
#pragma unroll
        for (int f = 0; f < N; ++f) fill(f);
      }
      unrolled<M>([&](auto nth) {
        constexpr int q = decltype(nth)::value;
        constexpr int r0 = reads_by<M, F, SPAN>(q);
        unrolled<reads_by<M, F, SPAN>(q + 1) - r0>([&](auto r) {
          reads(std::integral_constant<int, r0 + decltype(r)::value>{});
        });
        f32x4& c = acc[O.i[q]][O.j[q]];
        const s16x8 w = wf[CUR][O.i[q]], a = af[CUR][O.j[q]];
        // Fill f is at product (2 f + 1) M / 2 N: at this one, if any.
        constexpr int f = q * N / M;
        constexpr bool here = N > 0 && (2 * f + 1) * M / (2 * (N + !N)) == q;
        if constexpr (here && decltype(joined)::value) {
          const FillSource v = from(f);
          mfma16_acc_fill<decltype(once)::value, Tag>(
              c, w, a, v.base, v.at,
              (uint32_t)(uintptr_t)(__attribute__((address_space(3)))
                                    void*)to,
              f * TP_FILL);
        } else {
          if constexpr (here) fill(f);
          mfma16_acc<Tag>(c, w, a);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    // Stage s fills weights of stage s + PW - 1 in its first step and rows of
    // stage s + PA in its second, as long as there are any; the wait between
    // them for the next stage leaves what was filled after it.
    constexpr int AHEAD_A = (PA - 1) * FW + (PA - 2) * FA;
    constexpr int AHEAD_W = (PW - 2) * (FA + FW);
    constexpr int AHEAD = AHEAD_A < AHEAD_W ? AHEAD_A : AHEAD_W;
    static_assert(AHEAD + FA < 64);
    constexpr int LAST = PA > PW - 1 ? PA : PW - 1;
#pragma unroll
    for (int t = -LAST - 1; t < 0; ++t) {
      if (t + PW - 1 >= 0 && t + PW - 1 < steps) {
#pragma unroll
        for (int i = 0; i < FW; ++i) fw(t + PW - 1, i, t + PW - 1);
      }
      if (t + PA >= 0 && t + PA < steps) {
#pragma unroll
        for (int i = 0; i < FA; ++i) fa(t + PA, i, t + PA);
      }
    }
    if constexpr (J > 0) {   // (behind the first fills)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      acc_fence(acc);
    }
    if (steps >= PW) lds_fill_wait<AHEAD + FA>();
    else lds_fill_wait();
    lds_barrier();
    unrolled<F>([&](auto r) { read(0, 0, 0, 0, r); });
    int ap = 0, wp = 0;
    // MORE: fills go on in the whole stage.
    auto stage = [&](const int s, auto more) {
      constexpr bool MORE = decltype(more)::value;
      constexpr std::integral_constant<int, 0> ZERO{};
      constexpr std::integral_constant<int, 1> ONE{};
      constexpr std::integral_constant<int, 3> THREE{};
      constexpr std::integral_constant<int, 4> FOUR{};
      const int an = ap == PA - 1 ? 0 : ap + 1;
      const int wn_ = wp == PW - 1 ? 0 : wp + 1, wl = wp == 0 ? PW - 1 : wp - 1;
      // (All reads well before the barrier, which waits for them.)
      step(ZERO, THREE, [&](auto r) { read(1, ap, wp, 1, r); },
           std::integral_constant<int, FW>{}, more,
           std::bool_constant<ONCE>{},
           [&](int f) { return from_w(s + PW - 1, f); }, w_to + wl * WB,
           [&](int f) {
             if (MORE || s + PW - 1 < steps) fw(s + PW - 1, f, wl);
           });
      // The next stage has landed when only what was filled after it is
      // under way; past the barrier no wave reads this one again.
      if constexpr (MORE) lds_fill_wait<AHEAD>();
      else wait_but<PW - 2>(steps - 2 - s);
      lds_barrier();
      step(ONE, FOUR, [&](auto r) { read(0, an, wn_, 0, r); },
           std::integral_constant<int, (MORE || LAST > PA ? FA : 0)>{}, more,
           std::false_type{}, [&](int f) { return from_a(s + PA, f); },
           a_to + ap * AB, [&](int f) {
             if (MORE || s + PA < steps) fa(s + PA, f, ap);
           });
      ap = an;
      wp = wn_;
    };
    int s = 0;
#pragma unroll 1
    for (; s + LAST < steps; ++s) stage(s, std::true_type{});
#pragma unroll 1
    for (; s < steps; ++s) stage(s, std::false_type{});
    if constexpr (J > 0) acc_fence(acc);
  }
};

}  // namespace vllm_amd
