// Which linear layers tile_linear.hip takes, and how.
#pragma once

#include <cstdint>

namespace vllm_amd {

// Weight rows of a tile (0: not one for that file) and parts of K.
struct TileForm { int cols, parts; };
TileForm tile_linear_form(int64_t M, int64_t rows_w, int64_t K, bool silu);

// Whether it is one for that file although stream_linear.hip takes it too.
inline bool tile_linear_first(int64_t M, int64_t rows_w, int64_t K,
                              bool silu) {
  return M > 32 && M <= 64 && tile_linear_form(M, rows_w, K, silu).cols > 0;
}

// What a workgroup takes, of m_tiles x n_tiles tiles with K in parts: each XCD
// (workgroups go round them) has a run of `run` jobs, in which those beside
// each other have weights in common, then columns of K. It begins `turn` stages
// of K into its part: the same for those of an XCD that share weights, another
// for others.
struct TileJob { int part, m_tile, n_tile, turn; };
constexpr TileJob tile_job(int xcd, int nth, int run, int m_tiles,
                           int n_tiles) {
  const int job = xcd * run + nth;
  const int weights = job / m_tiles;
  return {weights / n_tiles, job % m_tiles, weights % n_tiles,
          weights - xcd * run / m_tiles + xcd * 4};
}
// Stages of K of a part: it ends where the next begins.
constexpr int tile_part(int stages, int part, int parts) {
  return stages * part / parts;
}

}  // namespace vllm_amd
