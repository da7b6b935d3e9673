// Which linear layers tile_linear.hip takes, and how.
#pragma once

#include <cstdint>

namespace vllm_amd {

// Weight rows of a tile (0: not one for that file) and parts of K.
struct TileForm { int cols, parts; };
TileForm tile_linear_form(int64_t M, int64_t rows_w, int64_t K, bool silu);

}  // namespace vllm_amd
