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

}  // namespace vllm_amd
