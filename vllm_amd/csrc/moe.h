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
// row tiles that hold rows, one part of each per XCD. There the row tiles of
// an expert, in equal groups of at most eight, go through the column blocks
// together: those beside each other share weights, and the blocks rows, in its
// L2. ms, groups of eight that end anywhere in an expert and these: 64 experts
// of 7168 x 2048, 8 a token, 4096 tokens 2.75 and 2.66, 1600 unevenly 1.53 and
// 1.42; 128 of 2048 x 768, 512 tokens 0.253 and 0.243; 8 of 4096 x 14336, 2 a
// token, 4096 tokens 2.41 and 2.33. Where a part has eight row tiles at most
// they are one group (the same 8 experts, 400 tokens, a tile each: 0.606, one
// expert after another 0.633).
constexpr int TILE_GROUP = 8;
struct TilePart { int m0, m1, n0, n1; };   // of an XCD
inline __host__ __device__ TilePart tile_part_of(int xcd, int tiles,
                                                 int n_blocks, int split) {
  const int parts = 8 / split, y = xcd / split, c = xcd % split;
  return {tiles * y / parts, tiles * (y + 1) / parts, n_blocks * c / split,
          n_blocks * (c + 1) / split};
}
// Tile q of those of a run of row tiles of one expert, from `first` on.
inline __host__ __device__ void tile_of_run(int first, int tiles, int blocks,
                                            int q, int& m, int& n) {
  const int groups = (tiles + TILE_GROUP - 1) / TILE_GROUP;
  // Group g begins at row tile tiles * g / groups.
  const int at = q / blocks;   // a row tile of the group
  const int g = ((at + 1) * groups - 1) / tiles;
  const int r0 = tiles * g / groups;
  const int rows = tiles * (g + 1) / groups - r0;
  m = first + r0 + (q - r0 * blocks) % rows;
  n = (q - r0 * blocks) / rows;
}
DEVINL bool tile_of_block(const int* __restrict__ expert_tiles, int tiles,
                          int n_blocks, int split, int& m, int& n) {
  const TilePart p =
      tile_part_of((int)blockIdx.x & 7, tiles, n_blocks, split);
  const int blocks = p.n1 - p.n0;
  const int l = (int)blockIdx.x >> 3;
  if (l >= (p.m1 - p.m0) * blocks) return false;
  if (p.m1 - p.m0 <= TILE_GROUP) {
    tile_of_run(p.m0, p.m1 - p.m0, blocks, l, m, n);
    n += p.n0;
    return true;
  }
  // The run that row tile `at` is in: 32 to either side come at once.
  const int at = p.m0 + l / blocks;
  const int lane = threadIdx.x % WAVE_SIZE;
  const int near = at - 32 + lane;
  const int it = expert_tiles[min(max(near, p.m0), p.m1 - 1)];
  const int expert = __builtin_amdgcn_readlane(it, 32);
  const uint64_t other =
      __ballot(near < p.m0 || near >= p.m1 || it != expert);
  // (A bit behind the 32 to either side ends the count. As a select of 32
  // where there is none, the compiler had it read another compare's
  // condition: tests/test_conditions.py.)
  const uint64_t low = other << 32, high = other >> 32;
  int first = at - __builtin_clzll(low | 1ull << 31);
  int end = at + __builtin_ctzll(high | 1ull << 32);
  for (bool more = low == 0; more && first > p.m0; ) {
    const int i = first - 1 - lane;
    const uint64_t o =
        __ballot(i < p.m0 || expert_tiles[max(i, p.m0)] != expert);
    first -= o ? __builtin_ctzll(o) : WAVE_SIZE;
    more = o == 0;
  }
  for (bool more = high == 0; more; ) {
    const int i = end + lane;
    const uint64_t o =
        __ballot(i >= p.m1 || expert_tiles[min(i, p.m1 - 1)] != expert);
    end += o ? __builtin_ctzll(o) : WAVE_SIZE;
    more = o == 0;
  }
  tile_of_run(first, end - first, blocks, l - (first - p.m0) * blocks, m, n);
  n += p.n0;
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
