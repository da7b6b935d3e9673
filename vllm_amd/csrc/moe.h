// What the grouped expert products of moe.hip and moe_tiles.hip share.
#pragma once

#include "common.h"

namespace vllm_amd {

namespace moe {

// What the epilogue of a product does.
enum Act { NONE = 0, SILU_GATED = 1, RELU2 = 2 };

DEVINL float silu_mul(float g, float u) { return g / (1.f + __expf(-g)) * u; }
DEVINL float relu2(float x) {
  const float r = fmaxf(x, 0.f);
  return r * r;
}

// Which (row tile, column block) a workgroup takes; every eighth workgroup
// runs on the same XCD. Streamed weights: each XCD takes a run of
// neighbours in (column block, row tile) order.
DEVINL bool tile_of_block(int m_tiles, int n_blocks, int& m, int& n) {
  const int total = m_tiles * n_blocks;
  const int per = (total + 7) / 8;
  const int l = (int)blockIdx.x >> 3;
  const int p = ((int)blockIdx.x & 7) * per + l;
  if (l >= per || p >= total) return false;
  m = p % m_tiles;
  n = p / m_tiles;
  return true;
}
// Tiles: `split` parts of the column blocks times 8 / split parts of the
// row tiles that hold rows, one part of each per XCD; eight row tiles by
// some column blocks run there at a time, so tiles of an expert share
// weights and blocks share rows in its L2.
DEVINL bool tile_of_block(int tiles, int n_blocks, int split, int& m,
                          int& n) {
  constexpr int GROUP = 8;
  const int x = (int)blockIdx.x & 7;
  const int l = (int)blockIdx.x >> 3;
  const int parts = 8 / split, y = x / split, c = x % split;
  const int m0 = tiles * y / parts, mm = tiles * (y + 1) / parts - m0;
  const int n_lo = n_blocks * c / split;
  const int nn = n_blocks * (c + 1) / split - n_lo;
  if (l >= mm * nn) return false;
  const int g = l / (GROUP * nn), q = l - g * (GROUP * nn);
  const int rows = min(GROUP, mm - g * GROUP);
  m = m0 + g * GROUP + q % rows;
  n = n_lo + q / rows;
  return true;
}

// Rows of this tile that hold a (token, slot) pair: they come first.
template <int TM>
DEVINL int rows_of_tile(const int* __restrict__ sorted, int tile,
                        int total_flat) {
  int n = 0;
#pragma unroll
  for (int i = 0; i < TM; i += WAVE_SIZE)
    n += __popcll(__ballot(
        sorted[tile * TM + i + (threadIdx.x % WAVE_SIZE)] < total_flat));
  return n;
}

constexpr int TL_W = 256;   // weight rows of a tile

// Products in 128- (form 1) or 256-row tiles (form 2), moe_tiles.hip; the
// operands as run_gemm has checked them.
struct TileArgs {
  const short* a;
  int64_t lda;
  const short* w;
  int64_t expert_stride;
  short* c;
  int64_t ldc;
  const int* sorted;
  const int* expert_tiles;
  int K, N, topk_div, total_flat, m_tiles, n_blocks, split;
};
void launch_tiles(const TileArgs& t, int form, int act, bool bf16,
                  unsigned blocks, hipStream_t stream);

}  // namespace moe

}  // namespace vllm_amd
