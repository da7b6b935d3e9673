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
// of 7168 x 2048, 8 a token, 4096 tokens 2.70 and 2.65, 1600 unevenly 1.58 and
// 1.45; 128 of 2048 x 768, 512 tokens 0.267 and 0.260; 8 of 4096 x 14336, 2 a
// token, 1700 tokens 1.30 and 1.22, 4096 2.40 and 2.37.
//
// Where a part has eight row tiles at most they are one group (the same 8
// experts, 400 tokens, a tile each: 0.606, one expert after another 0.633). Nor
// do groups end with their experts where an XCD has all of 16 tiles of 128 rows
// or fewer: experts of one tile and of two, side by side, wait for weights and
// multiply at the same time. Of these 8 experts with 330 to 740 tokens (9 to 16
// tiles, 32 samples), groups that end with their experts took 1.9 % more on
// average, from 3.7 % less to 6.2 % more (0.670 and 0.712). With tiles of 256 rows
// they gain 1.3 % from 12 tiles on, and with fewer it is even (-3 to 3 %); as
// many experts as tiles have nothing to mix (16 of 5120 x 8192, 1 a token, 1000
// tokens 0.769 and 0.752).
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
// Tile l of a part. expert_of(i): of row tile i; ballot(f): the lanes of a wave
// that f(lane) is true for, of a device's or the host's. few: the part has all
// row tiles, of 128 rows.
template <typename Expert, typename Ballot>
inline __host__ __device__ void tile_of_part(const TilePart& p, bool few,
                                             int l, const Expert& expert_of,
                                             const Ballot& ballot, int& m,
                                             int& n) {
  const int tiles = p.m1 - p.m0, blocks = p.n1 - p.n0;
  int first = p.m0, end = p.m1;
  if (tiles > TILE_GROUP) {
    if (few && tiles <= 2 * TILE_GROUP && ballot([&](int lane) {
          const int i = p.m0 + (lane < tiles - 1 ? lane : tiles - 2);
          return expert_of(i) == expert_of(i + 1);
        })) {
      // (Eight and the rest. In two halves 14 tiles lost 3 %.)
      const int g = l / (TILE_GROUP * blocks), q = l % (TILE_GROUP * blocks);
      first += g * TILE_GROUP;
      const int rows = end - first < TILE_GROUP ? end - first : TILE_GROUP;
      m = first + q % rows;
      n = p.n0 + q / rows;
      return;
    }
    // The run that row tile `at` is in: 32 to either side come at once.
    const int at = p.m0 + l / blocks;
    const int expert = expert_of(at);
    auto others = [&](int from, int step) -> uint64_t {
      return ballot([&](int lane) {
        const int i = from + lane * step;
        const int in = i < p.m0 ? p.m0 : i < p.m1 ? i : p.m1 - 1;
        const bool other = expert_of(in) != expert;   // (no branch)
        return (i != in) | other;
      });
    };
    const uint64_t near = others(at - 32, 1);
    // (A bit behind the 32 to either side ends the count. As a select of 32
    // where there is none, the compiler had it read another compare's
    // condition: tests/test_conditions.py.)
    const uint64_t low = near << 32, high = near >> 32;
    first = at - __builtin_clzll(low | 1ull << 31);
    end = at + __builtin_ctzll(high | 1ull << 32);
    for (bool more = low == 0; more;) {
      const uint64_t o = others(first - 1, -1);
      first -= o ? __builtin_ctzll(o) : WAVE_SIZE;
      more = o == 0;
    }
    for (bool more = high == 0; more;) {
      const uint64_t o = others(end, 1);
      end += o ? __builtin_ctzll(o) : WAVE_SIZE;
      more = o == 0;
    }
  }
  tile_of_run(first, end - first, blocks, l - (first - p.m0) * blocks, m, n);
  n += p.n0;
}
template <int TM>
DEVINL bool tile_of_block(const int* __restrict__ expert_tiles, int tiles,
                          int n_blocks, int split, int& m, int& n) {
  const TilePart p =
      tile_part_of((int)blockIdx.x & 7, tiles, n_blocks, split);
  const int l = (int)blockIdx.x >> 3;
  if (l >= (p.m1 - p.m0) * (p.n1 - p.n0)) return false;
  tile_of_part(
      p, TM == 128 && split == 8, l,
      [&](int i) { return expert_tiles[i]; },
      [&](auto f) { return __ballot(f((int)threadIdx.x % WAVE_SIZE)); }, m, n);
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
