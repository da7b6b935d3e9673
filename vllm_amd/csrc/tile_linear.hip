// Linear layers on 65 to 256 rows, where one workgroup holds all rows of a
// tile of columns (gfx950): out[M, N] = x[M, K] @ w[N, K]^T, and the same
// with silu(gate) * up of two halves of w as the epilogue.
//
// Between bound by the weights' way from HBM and by the matrix cores
// (tile_product.h). Weights are read by one workgroup only and leave L2 first;
// x stays. Nothing splits K here: partial sums of so many rows cost what the
// split gains. So a layer must have nearly as many tiles as CUs run, or a
// multiple of that, to be ahead of the tuned library (tile_form below).
// us, library (and activation) -> this, weights from HBM:
//   28672 x 4096 with the activation, 80 rows 59 -> 47, 256 rows 73 -> 61;
//   22016 x 4096 with it, 192 rows 60 -> 54, 256 rows 64 -> 57; 129280 x 7168,
//   80 rows 345 -> 313, 256 rows 405 -> 385; 128256 x 4096, 256 rows 275 -> 251;
//   32000 x 4096, 80 rows 59 -> 52, 192 rows 67 -> 63.

#include <torch/all.h>
#include <c10/hip/HIPStream.h>

#include "tile_product.h"

namespace vllm_amd {

namespace {

constexpr int TI_ROWS = 256;

// N: columns of out. SILU: w has 2N rows, gate then up; a wave's gate rows,
// then the up rows of the same columns.
template <typename Tag, bool SILU, int WGM, int NI, int MI, int PA, int PW>
__global__ __launch_bounds__(TP_THREADS, 1) void tile_linear_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const short* __restrict__ w, const int M, const int N, const int K,
    const int tiles) {
  using P = TileProduct<Tag, WGM, NI, MI, PA, PW>;
  __shared__ __align__(16) char lds[P::LDS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l32 = lane & 31;
  const int half = lane >> 5;
  constexpr int NO = SILU ? NI / 2 : NI;
  // Each XCD (workgroups go round them) takes a run of tiles.
  const int run = (tiles + 7) / 8;
  const int tile = blockIdx.x % 8 * run + blockIdx.x / 8;
  if (blockIdx.x / 8 >= run || tile >= tiles) return;
  const int n0 = tile * (P::TN / (SILU ? 2 : 1));
  const short* wt = w + (int64_t)n0 * K;

  // Byte places of this lane's pieces; rows past the end repeat the last.
  uint32_t ap[P::FA], wp[P::FW];
#pragma unroll
  for (int i = 0; i < P::FA; ++i) {
    const int r = (wave * P::FA + i) * 8 + (lane >> 3);
    ap[i] = (uint32_t)min(r, M - 1) * (uint32_t)(K * 2) +
            ((lane & 7) ^ tp_swap(r)) * 16;
  }
#pragma unroll
  for (int i = 0; i < P::FW; ++i) {
    const int r = (wave * P::FW + i) * 8 + (lane >> 3);
    int src;
    if constexpr (SILU)
      src = min(r / P::WW * (P::WW / 2) + r % (P::WW / 2), N - 1 - n0) +
            r / (P::WW / 2) % 2 * N;
    else
      src = min(r, N - 1 - n0);
    wp[i] = (uint32_t)src * (uint32_t)(K * 2) +
            ((lane & 7) ^ tp_swap(r)) * 16;
  }
  P::run(
      lds, K / TP_K, M,
      [&](int s, int i, char* dst) { lds_fill16(x + s * TP_K, ap[i], dst); },
      [&](int s, int i, char* dst) {
        lds_fill16_once(wt + s * TP_K, wp[i], dst);
      },
      [&](auto n, auto& acc) {
        constexpr int J = decltype(n)::value;
        const int wm = wave / P::WGN, wn = wave % P::WGN;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int row = (j * WGM + wm) * 32 + l32;
          if (row >= M) continue;
          short* o = out + (int64_t)row * N;
#pragma unroll
          for (int i = 0; i < NO; ++i) {
            f32x16 v = acc[i][j];
            const int c0 = n0 + (wn * NO + i) * 32;
            if constexpr (SILU) {
#pragma unroll
              for (int r = 0; r < 16; ++r)
                v[r] = v[r] / (1.f + __expf(-v[r])) * acc[i + NI / 2][j][r];
            }
#pragma unroll
            for (int b = 0; b < 4; b += 2) {
              const i32x4 chunk = row_chunk<Tag>(v, b);
              const int col = c0 + b * 8 + half * 8;
              if (col < N) *reinterpret_cast<i32x4*>(o + col) = chunk;
            }
          }
        }
      });
}

// 0: the library; else 128 or 256 weight rows a tile, for M rows by rows_w
// weight rows of K.
//
// The share of its rounds over 256 CUs that a form keeps busy decides: 256
// where that is at least 95 % (for up to 128 rows of a plain product in more
// than one round: 65536 x 4096 alone, 80 rows, 128 us, the library 124), else
// 128 where that is one round. An activation, which saves a launch and a pass,
// makes up for a third of one round, or a tenth of several. us, this and the
// library: 28672 x 4096, 128 rows, 224 tiles of 128: 57.4 and 57.2; 65536 x
// 4096, 128 rows, 512 tiles of 128: 136 and 125; 57344 x 4096 with the
// activation, 128 rows, 448 tiles: 118 and 102; 152064 x 3584, 256 rows, 594
// tiles of 256: 288 and 259.
//
// Plain products whose K is at most eight times their rows write too much
// beside what they read, and workgroups that end together wait for it. us, this
// and the library: 65536 x 512, 256 rows 30.0 and 24.5, x 1024 39.7 and 37.9, x
// 2048 73 and 76; 128256 x 256, 128 rows 30.6 and 26.2, x 1024 61.5 and 60.0,
// 65 rows 54 and 62. An activation halves what is written.
int tile_form(int64_t M, int64_t rows_w, int64_t K, bool silu) {
  if (M <= 64 || M > TI_ROWS || (!silu && K <= 8 * M)) return 0;
  auto rounds = [&](int tile) { return (rows_w + tile * 256 - 1) / tile / 256; };
  auto busy = [&](int tile) {
    return (double)((rows_w + tile - 1) / tile) / (double)(rounds(tile) * 256);
  };
  if (busy(256) >= 0.95 && (silu || M > 128 || rounds(256) > 1)) return 256;
  const double least = rounds(128) > 1 ? (silu ? 0.9 : 2.) : silu ? 0.65 : 0.95;
  return busy(128) >= least ? 128 : 0;
}

template <typename Tag, bool SILU>
void launch(torch::Tensor& out, const torch::Tensor& x,
            const torch::Tensor& w, int form) {
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)out.size(1);
  const int tiles = ceil_div(N, form / (SILU ? 2 : 1));
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(ceil_div(tiles, 8) * 8), dim3(TP_THREADS),
                       0, c10::hip::getCurrentHIPStream().stream(),
                       (short*)out.data_ptr(), (const short*)x.data_ptr(),
                       (const short*)w.data_ptr(), M, N, K, tiles);
  };
  if (M <= 128) {
    if (form == 128) go(tile_linear_kernel<Tag, SILU, 2, 2, 2, 5, 5>);
    else             go(tile_linear_kernel<Tag, SILU, 1, 2, 4, 3, 3>);
  } else {
    if (form == 128) go(tile_linear_kernel<Tag, SILU, 2, 2, 4, 3, 3>);
    else             go(tile_linear_kernel<Tag, SILU, 2, 4, 4, 2, 3>);
  }
}

}  // namespace

// The form for a product of these sizes, 0 if it is not one for this file.
int tile_linear_form(int64_t M, int64_t rows_w, int64_t K, bool silu) {
  if (rows_w <= 0 || rows_w % (silu ? 16 : 8) != 0 || K <= 0 ||
      K % TP_K != 0 || K >= (1 << 22) || (rows_w + 256) * K * 2 >= (1ll << 32))
    return 0;
  return tile_form(M, rows_w, K, silu);
}

// The product of x [M, K] and w [rows, K], both contiguous, into out [M, n],
// if it is one that this file takes.
bool tile_linear(torch::Tensor& out, const torch::Tensor& x,
                 const torch::Tensor& w, bool silu) {
  const int64_t K = x.size(1);
  const int form = tile_linear_form(x.size(0), w.size(0), K, silu);
  if (form == 0 || w.size(1) != K || w.scalar_type() != x.scalar_type() ||
      (x.scalar_type() != torch::kBFloat16 &&
       x.scalar_type() != torch::kHalf) ||
      !x.is_contiguous() || !w.is_contiguous() ||
      (uintptr_t)x.data_ptr() % 16 != 0 || (uintptr_t)w.data_ptr() % 16 != 0)
    return false;
  if (x.scalar_type() == torch::kBFloat16) {
    if (silu) launch<BF16Tag, true>(out, x, w, form);
    else      launch<BF16Tag, false>(out, x, w, form);
  } else {
    if (silu) launch<FP16Tag, true>(out, x, w, form);
    else      launch<FP16Tag, false>(out, x, w, form);
  }
  HIP_CHECK_KERNEL();
  return true;
}

}  // namespace vllm_amd
