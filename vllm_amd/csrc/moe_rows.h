// Up to 64 rows of an expert past its weights as they stream in: moe.hip, and
// moe_tiles.hip for tiles that hold no more.
#pragma once

#include "moe.h"
#include "stream_product.h"

namespace vllm_amd {

namespace moe {

constexpr int SR_WIDE = 128, SR_NARROW = 32;   // weight rows of a workgroup
constexpr int ROWS_LDS = 160 * 1024;

// Rows row0 .. row0 + rows - 1 in tile order by NI * 16 weight rows (gated:
// half of them gate rows, half the up rows of the same columns) from n0 on;
// four waves, of which WV multiply.
template <typename Tag, int ACT, int NI, int XG, int WV, int D>
DEVINL void stream_rows(char* lds, const short* __restrict__ A,
                        const short* __restrict__ W, short* __restrict__ C,
                        int64_t ldc, const int* __restrict__ sorted, int K,
                        int N, int topk_div, int row0, int rows, int n0) {
  using P = StreamProduct<Tag, NI, XG, WV, D>;
  constexpr bool GATED = ACT == SILU_GATED;
  constexpr int NO = NI / (GATED ? 2 : 1);   // 16-column groups
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  uint32_t wat[2 * NI], xat[XG];
#pragma unroll
  for (int i = 0; i < 2 * NI; ++i) {
    const int r = i * 8 + (lane >> 3);
    const int up = r >= NO * 16 ? 1 : 0;
    wat[i] = sp_place(min(r - up * NO * 16, N - 1 - n0) + up * N, r, K);
  }
#pragma unroll
  for (int i = 0; i < XG; ++i) {
    const int lr = i * 8 + (lane >> 3);
    const int r = row0 + min(lr, rows - 1);
    xat[i] = sp_place(topk_div > 0 ? sorted[r] / topk_div : r, lr, K);
  }
  P::run(lds, wave, 0, K / SP_K, blockIdx.x / 8,
         reinterpret_cast<const char*>(W + (int64_t)n0 * K), wat,
         reinterpret_cast<const char*>(A), xat);
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
#pragma unroll
  for (int u = 0; u < (NO * P::MT + 3) / 4; ++u) {
    const int t = u * 4 + wave;
    if (t >= NO * P::MT) break;
    f32x4 v = P::sum(lds, t);
    if constexpr (GATED) {
      const f32x4 up = P::sum(lds, NO * P::MT + t);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = silu_mul(v[r], up[r]);
    } else if constexpr (ACT == RELU2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = relu2(v[r]);
    }
    const int row = t % P::MT * 16 + l16;
    const int col = n0 + t / P::MT * 16 + l4 * 4;
    if (row < rows && col < N && (XG > 1 || l16 < 8))
      *reinterpret_cast<int2*>(C + (int64_t)(row0 + row) * ldc + col) =
          int2{pack2<Tag>(v[0], v[1]), pack2<Tag>(v[2], v[3])};
  }
}

// The same, with as many steps on the way as LDS holds. Called by all threads
// of a workgroup of four waves; a second call needs a barrier before it.
template <typename Tag, int ACT, int NI>
DEVINL void rows_body(char* lds, const short* __restrict__ A,
                      const short* __restrict__ W, short* __restrict__ C,
                      int64_t ldc, const int* __restrict__ sorted, int K,
                      int N, int topk_div, int row0, int rows, int n0) {
  auto go = [&](auto xg, auto wv, auto d) {
    constexpr int XG = decltype(xg)::value, WV = decltype(wv)::value,
                  D = decltype(d)::value;
    static_assert(StreamProduct<Tag, NI, XG, WV, D>::LDS <= ROWS_LDS);
    stream_rows<Tag, ACT, NI, XG, WV, D>(lds, A, W, C, ldc, sorted, K, N,
                                         topk_div, row0, rows, n0);
  };
  constexpr bool WIDE = NI == SR_WIDE / 16;
  using one = std::integral_constant<int, 1>;
  using two = std::integral_constant<int, 2>;
  using four = std::integral_constant<int, 4>;
  using depth = std::integral_constant<int, WIDE ? 2 : 4>;
  if (rows <= 8)       go(one{}, four{}, depth{});
  else if (rows <= 16) go(two{}, four{}, depth{});
  else if (rows <= 32) go(four{}, four{}, depth{});
  else                 go(std::integral_constant<int, 8>{},
                          std::integral_constant<int, WIDE ? 2 : 4>{},
                          std::integral_constant<int, 3>{});
}

}  // namespace moe

}  // namespace vllm_amd
