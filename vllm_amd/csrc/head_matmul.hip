// Per-head matrix product for MI355X (gfx950):
//   out[t, h, :] = x[t, h, :] @ W[h]        x [T, H, K], W [H, K, N]
// 16-bit operands, fp32 sums (the products of 16-bit values are exact in
// fp32, so this is the fp32 product of the same operands). It carries MLA
// queries into the latent space and attention results out of it.
//
// Small T is bound by reading W once (16.8 MB at 128 heads of 128 x 512),
// large T by writing the wide side; in between the operands are small, so
// a plain tile does: one workgroup is 64 tokens x 128 columns of a head,
// W goes to LDS in steps of 128 rows, filled straight from global memory:
// one step is all of it (then five workgroups fit a CU), four are all on
// their way at once while there is a CU for each workgroup, and else two
// alternate. Each of four waves takes 32 tokens x 64 columns, which
// balances LDS reads against loads of x. The product is formed transposed
// (W^T x^T): W^T fragments are transposing LDS reads of the row-major
// tile, x^T fragments plain 16 B loads of token rows, and a lane ends up
// with four neighbouring columns of one token, eight after a trade between
// two tiles (16 B stores: 9 % faster than 8 B ones).
// Against widening both operands and a library fp32 product, us for
// 128 heads of 128 x 512: 128 tokens 121 -> 12; 3901 tokens 1073 -> 274. Two
// alternating steps in every case: 128 x 512, 128 tokens 13.6, now 12.2, 256
// 21.8, now 19.7; 512 x 128, 8 tokens 8.3, now 7.6, 128 11.4, now 10.6.

#include <torch/all.h>
#include <c10/hip/HIPStream.h>

#include "common.h"

namespace vllm_amd {

namespace {

constexpr int HM_M = 64;      // tokens per workgroup
constexpr int HM_N = 128;     // columns per workgroup
constexpr int HM_K = 128;     // rows of W per LDS tile
constexpr int HM_THREADS = 256;
constexpr int HM_DEEP = 256;  // workgroups: one a CU
constexpr int HM_TILE = HM_K * HM_N * 2;                   // bytes
constexpr int HM_FILL = HM_TILE / 16 / HM_THREADS;

DEVINL int hm_swap(int row) { return (row & 3) | ((row >> 1) & 4); }

// BUFS 1 and 4: K is that many tiles, and all of them are on their way at
// once; 2: any number, alternating.
template <typename Tag, int BUFS>
__global__ __launch_bounds__(HM_THREADS, BUFS == 1 ? 4 : 4 / BUFS)
    void head_matmul_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const short* __restrict__ w, const int T, const int H, const int K,
    const int N, const int64_t x_row, const int64_t x_head) {
  __shared__ __align__(16) char lds[BUFS * HM_TILE];
  const int n0 = blockIdx.x * HM_N;
  const int h = blockIdx.y;
  const int t0 = blockIdx.z * HM_M;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  const int mw = (wave & 1) * 32;    // tokens and columns of this wave
  const int nw = (wave >> 1) * 64;

  // 32 B segments of a row are exchanged by the row, so that the eight
  // rows a transposing read takes per half wave (0..3 and 8..11, or 4
  // further on) lie on different banks.
  const short* wt = w + (int64_t)h * K * N + n0;
  auto fill = [&](int k0, int buf) {
#pragma unroll
    for (int i = 0; i < HM_FILL; ++i) {
      const int c = (wave * HM_FILL + i) * WAVE_SIZE + lane;
      const int r = c >> 4;
      const int s = (((c & 15) >> 1) ^ hm_swap(r)) * 2 + (c & 1);
      lds_fill16(wt + (int64_t)(k0 + r) * N + s * 8,
                 lds + buf * HM_TILE + (wave * HM_FILL + i) * WAVE_SIZE * 16);
    }
  };
  const short* xr[2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
    xr[m] = x + (int64_t)min(t0 + mw + m * 16 + l16, T - 1) * x_row +
            h * x_head + l4 * 8;

  f32x4 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int m = 0; m < 2; ++m) acc[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int r = l4 * 8 + (l16 >> 2);   // row of this lane's reads, mod 32
  s16x8 xf[BUFS == 4 ? 4 : 1][HM_K / 32][2];
  auto load_x = [&](int k0, s16x8 (&to)[HM_K / 32][2]) {
#pragma unroll
    for (int kk = 0; kk < HM_K / 32; ++kk)
#pragma unroll
      for (int m = 0; m < 2; ++m)
        to[kk][m] = *reinterpret_cast<const s16x8*>(xr[m] + k0 + kk * 32);
  };
  auto multiply = [&](int buf, const s16x8 (&xs)[HM_K / 32][2]) {
    const char* t = lds + buf * HM_TILE;
#pragma unroll
    for (int kk = 0; kk < HM_K / 32; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int seg = (nw >> 4) + i;
        const char* at = t + (kk * 32 + r) * (HM_N * 2) +
                         (seg ^ hm_swap(r)) * 32 + (l16 & 3) * 8;
        const s16x4 a = lds_read_tr(at);
        const s16x4 b = lds_read_tr(at + 4 * (HM_N * 2));
        const s16x8 wf = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[i][m] = mfma16<Tag>(wf, xs[kk][m],
                                                            acc[i][m]);
      }
  };
  if constexpr (BUFS == 2) {
    fill(0, 0);
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += HM_K, buf ^= 1) {
      load_x(k0, xf[0]);
      lds_fill_wait();
      __syncthreads();
      if (k0 + HM_K < K) fill(k0 + HM_K, buf ^ 1);
      multiply(buf, xf[0]);
    }
  } else {
#pragma unroll
    for (int s = 0; s < BUFS; ++s) load_x(s * HM_K, xf[s]);
#pragma unroll
    for (int s = 0; s < BUFS; ++s) fill(s * HM_K, s);
#pragma unroll
    for (int s = 0; s < BUFS; ++s) {
      if (s == 0)      lds_fill_wait<(BUFS - 1) * HM_FILL>();
      else if (s == 1) lds_fill_wait<(BUFS > 2 ? BUFS - 2 : 0) * HM_FILL>();
      else if (s == 2) lds_fill_wait<HM_FILL>();
      else             lds_fill_wait();
      lds_barrier();
      multiply(s, xf[s]);
    }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int tok = t0 + mw + m * 16 + l16;
    if (tok >= T) continue;
    // Tiles i and i + 1 have columns l4*4 .. + 3 here; neighbouring l4
    // trade halves, so that a lane stores eight columns of one of them.
    short* o = out + ((int64_t)tok * H + h) * N + n0 + nw + (l4 & 1) * 16 +
               (l4 >> 1) * 8;
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const auto s0 = __builtin_amdgcn_permlane16_swap(
          pack2<Tag>(acc[i][m][0], acc[i][m][1]),
          pack2<Tag>(acc[i + 1][m][0], acc[i + 1][m][1]), false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(
          pack2<Tag>(acc[i][m][2], acc[i][m][3]),
          pack2<Tag>(acc[i + 1][m][2], acc[i + 1][m][3]), false, false);
      const int a0 = s0[0], a1 = s1[0], b0 = s0[1], b1 = s1[1];
      *reinterpret_cast<i32x4*>(o + i * 16) = i32x4{a0, a1, b0, b1};
    }
  }
}

}  // namespace

// x [T, H, K] (rows and heads may be strided, 16 B aligned), w [H, K, N].
torch::Tensor head_matmul(torch::Tensor x, torch::Tensor w) {
  TORCH_CHECK(x.dim() == 3 && w.dim() == 3 && x.size(1) == w.size(0) &&
              x.size(2) == w.size(1), "head_matmul: [T, H, K] x [H, K, N]");
  TORCH_CHECK(x.scalar_type() == w.scalar_type() &&
              (x.scalar_type() == torch::kBFloat16 ||
               x.scalar_type() == torch::kHalf), "head_matmul: bf16/fp16 only");
  TORCH_CHECK(w.is_contiguous() && x.stride(2) == 1 &&
              x.stride(0) % 8 == 0 && x.stride(1) % 8 == 0 &&
              (uintptr_t)x.data_ptr() % 16 == 0 &&
              (uintptr_t)w.data_ptr() % 16 == 0,
              "head_matmul: rows must be 16 B aligned");
  const int T = (int)x.size(0), H = (int)x.size(1), K = (int)x.size(2);
  const int N = (int)w.size(2);
  TORCH_CHECK(K % HM_K == 0 && N % HM_N == 0,
              "head_matmul: K and N must be multiples of 128");
  auto out = torch::empty({T, H, N}, x.options());
  if (T == 0) return out;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  dim3 grid(N / HM_N, H, ceil_div(T, HM_M));
  auto launch = [&](auto tag, auto bufs) {
    using Tag = decltype(tag);
    hipLaunchKernelGGL((head_matmul_kernel<Tag, decltype(bufs)::value>), grid,
                       dim3(HM_THREADS), 0, stream, (short*)out.data_ptr(),
                       (const short*)x.data_ptr(), (const short*)w.data_ptr(),
                       T, H, K, N, x.stride(0), x.stride(1));
  };
  auto by_tiles = [&](auto tag) {
    const int64_t groups = (int64_t)grid.x * grid.y * grid.z;
    if (K == HM_K)
      launch(tag, std::integral_constant<int, 1>{});
    else if (K == 4 * HM_K && groups <= HM_DEEP)
      launch(tag, std::integral_constant<int, 4>{});
    else
      launch(tag, std::integral_constant<int, 2>{});
  };
  if (x.scalar_type() == torch::kBFloat16) by_tiles(BF16Tag{});
  else by_tiles(FP16Tag{});
  HIP_CHECK_KERNEL();
  return out;
}

}  // namespace vllm_amd
