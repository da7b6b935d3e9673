// Grouped expert products for experts of many rows (gfx950): 128 or 256 x
// 256 tiles of tile_product.h, the matrix cores bound them. The product is
// formed transposed (weight rows are the A operand), so a lane ends up with
// four neighbouring columns of one row, eight after a trade with another
// quarter of the wave (16 B stores). Gated experts: a tile is 128 gate rows and
// the up rows of the same columns, a wave's gate groups before its up groups,
// and the activation is the epilogue.
//
// Tiles of at most 128 rows (what is left of an expert after whole tiles,
// or experts of few rows) lay the four waves out along the weights; 32-row
// groups without a row are left out.
//
// An expert that has at most 32 rows in all is no tile: its weights stream
// past them (moe_rows.h; a few rows after whole tiles meet their weights in
// L2 and stay a tile). Beside larger ones, us without and so: 64 experts of
// 7168 x 2048, 8 a token, 100 tokens (0 to 46 rows) 987 / 854, 300 (4 to 139)
// 1114 / 1031; 8 of 4096 x 14336, 2 a token, 100 tokens (15 to 41) 572 / 523.
// With up to 64 rows 906, 1086 and 594.
//
// 64 experts of 7168 x 2048, 4096 tokens of 8, 50 to 1925 rows an expert:
// 1.76 + 0.95 ms (eight waves by halves in turn 2.01 + 1.10); 512 rows each
// 1.47 + 0.84 (1.31 and 1.14 PFLOP/s: the second, of 32 stages, pays the start
// and end of its tiles; by products of 32 x 32 x 16 1.50 + 0.86). What uneven
// rows cost beyond their padding is weights read twice: tiles of an expert that
// are not in step do not meet in L2 (8.3 GB instead of 4.1 in the first
// product).

#include <torch/all.h>
#include <c10/hip/HIPStream.h>

#include "moe_rows.h"
#include "tile_product.h"

namespace vllm_amd {

namespace moe {

// One tile by TileProduct; `row0` is its first row in tile order.
template <typename Tag, int ACT, int WGM, int NG, int MG, int PA>
DEVINL void tile_body(char* lds, const TileArgs& t, const short* w,
                      const int row0, const int rows, const int n0) {
  using P = TileProduct<Tag, WGM, NG, MG, PA, 3>;
  static_assert(P::TN == TL_W && P::WW * P::WGN == TL_W);
  constexpr bool GATED = ACT == SILU_GATED;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l16 = lane & 15;
  const int N = t.N;

  uint32_t ap[P::FA], wp[P::FW];   // byte places of this lane's pieces
#pragma unroll
  for (int i = 0; i < P::FA; ++i) {
    const int lr = (wave * P::FA + i) * 8 + (lane >> 3);
    const int r = row0 + min(lr, rows - 1);
    ap[i] = (uint32_t)(t.topk_div > 0 ? t.sorted[r] / t.topk_div : r) *
                (uint32_t)t.lda * 2 +
            ((lane & 7) ^ tp_swap(lr)) * 16;
  }
#pragma unroll
  for (int i = 0; i < P::FW; ++i) {
    const int r = (wave * P::FW + i) * 8 + (lane >> 3);
    int src;
    if constexpr (GATED)   // a wave's gate rows, their up rows
      src = min(n0 + r / P::WW * (P::WW / 2) + r % (P::WW / 2), N - 1) +
            r / (P::WW / 2) % 2 * N;
    else
      src = min(n0 + r, N - 1);
    wp[i] = (uint32_t)src * (uint32_t)t.K * 2 +
            ((lane & 7) ^ tp_swap(r)) * 16;
  }
  P::template run<false>(
      lds, t.K / TP_K, rows,
      [&](int s, int i) { return FillSource{t.a + s * TP_K, ap[i]}; },
      [&](int s, int i) { return FillSource{w + s * TP_K, wp[i]}; },
      [&](auto n, auto& acc) {
        constexpr int J = decltype(n)::value;
        constexpr int NO = GATED ? P::NI / 2 : P::NI;
        const int wm = wave / P::WGN, wn = wave % P::WGN;
        const int col0 = n0 + wn * NO * 16 + row_start16();
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int row = P::row_of(j, wm) + l16;
          if (row >= rows) continue;
          short* c = t.c + (int64_t)(row0 + row) * t.ldc;
#pragma unroll
          for (int i = 0; i < NO; i += 2) {
            f32x4 v[2];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float a = acc[i + h][j][r];
                if constexpr (GATED)
                  v[h][r] = silu_mul(a, acc[i + h + NO][j][r]);
                else
                  v[h][r] = ACT == RELU2 ? relu2(a) : a;
              }
            const i32x4 o = row_chunk16<Tag>(v[0], v[1]);
            const int col = col0 + i * 16;
            if (col < N) *reinterpret_cast<i32x4*>(c + col) = o;
          }
        }
      });
}

constexpr int TL_FEW = 32;   // rows of an expert that are no tile

template <typename Tag, int ACT, int TM>
__launch_bounds__(TP_THREADS, 1) __global__
void moe_tile_kernel(const TileArgs t) {
  int tile, blk;
  if (!tile_of_block<TM>(t.expert_tiles, t.expert_tiles[t.m_tiles],
                         t.n_blocks, t.split, tile, blk))
    return;
  using Whole = TileProduct<Tag, 2, 4, 4, 2, 3>;
  using Half = TileProduct<Tag, 1, 2, 4, 3, 3>;
  static_assert(Whole::TM == 256 && Half::TM == 128);
  static_assert(Whole::LDS <= ROWS_LDS && Half::LDS <= ROWS_LDS);
  __shared__ __align__(16) char lds[ROWS_LDS];
  const int rows = rows_of_tile<TM>(t.sorted, tile, t.total_flat);
  const int n0 = blk * (ACT == SILU_GATED ? TL_W / 2 : TL_W);
  const short* w = t.w + t.expert_tiles[tile] * t.expert_stride;
  if (rows <= TL_FEW &&
      (tile == 0 || t.expert_tiles[tile - 1] != t.expert_tiles[tile])) {
    constexpr int PER = SR_WIDE / (ACT == SILU_GATED ? 2 : 1);
    for (int n = n0; n < min(n0 + TL_W / SR_WIDE * PER, t.N); n += PER) {
      if (n > n0) __syncthreads();
      rows_body<Tag, ACT, SR_WIDE / 16>(lds, t.a, w, t.c, t.ldc, t.sorted,
                                        t.K, t.N, t.topk_div, tile * TM,
                                        rows, n);
    }
    return;
  }
  if constexpr (TM == 256) {
    if (rows > 128) {
      tile_body<Tag, ACT, 2, 4, 4, 2>(lds, t, w, tile * TM, rows, n0);
      return;
    }
  }
  tile_body<Tag, ACT, 1, 2, 4, 3>(lds, t, w, tile * TM, rows, n0);
}

void launch_tiles(const TileArgs& t, int form, int act, bool bf16,
                  unsigned blocks, hipStream_t stream) {
  auto launch = [&](auto tag, auto act_tag) {
    using Tag = decltype(tag);
    constexpr int ACT = decltype(act_tag)::value;
    if (form == 2)
      hipLaunchKernelGGL((moe_tile_kernel<Tag, ACT, 256>), dim3(blocks),
                         dim3(TP_THREADS), 0, stream, t);
    else
      hipLaunchKernelGGL((moe_tile_kernel<Tag, ACT, 128>), dim3(blocks),
                         dim3(TP_THREADS), 0, stream, t);
  };
  auto by_act = [&](auto tag) {
    if (act == SILU_GATED)
      launch(tag, std::integral_constant<int, SILU_GATED>{});
    else if (act == RELU2)
      launch(tag, std::integral_constant<int, RELU2>{});
    else
      launch(tag, std::integral_constant<int, NONE>{});
  };
  if (bf16) by_act(BF16Tag{});
  else      by_act(FP16Tag{});
}

}  // namespace moe

}  // namespace vllm_amd
