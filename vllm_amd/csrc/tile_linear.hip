// Linear layers on 33 to 1024 rows, by tiles of all rows or of 256 of them
// (gfx950): out[M, N] = x[M, K] @ w[N, K]^T, and for up to 256 rows the same
// with silu(gate) * up of two halves of w as the epilogue.
//
// Between bound by the weights' way from HBM and by what a CU takes in: rows of
// x come from L2 (100 GB/s a CU, alone), weights from HBM (23 GB/s a CU where
// all read, 5.9 TB/s), and where both come one waits for the other rather than
// beside it, however much is under way: 128 rows of x and 64 of weights a stage
// at 49 GB/s a CU (4.2 TB/s of weights), 256 and 64 at 59 (3.0), 256 and 128 at
// 58 (4.9), 128 and 128 at 46 (5.9).
//
//  * Weights that one workgroup reads leave L2 first; x stays.
//  * Workgroups begin at different stages of K, those of an XCD that share
//    weights at the same one (tile_job): rows whose stride is a power of two
//    meet on few channels otherwise. A window of some 60 stages, so that x
//    stays in L2. 128 rows of weights alone at K = 16384 5.4 -> 7.0 TB/s; 28672
//    x 4096 with the activation, 128 rows 57 -> 52 us.
//  * Layers with few tiles split K over workgroups until about one a CU runs,
//    if K is long enough for the partial sums not to cost what that gains
//    (by_estimate below); a second launch adds them.
// us, library (and activation) -> this, weights from HBM:
//   28672 x 4096 with the activation, 80 rows 59 -> 46, 256 rows 84 -> 66;
//   22016 x 4096 with it, 192 rows 60 -> 54, 256 rows 64 -> 57; 128256 x 4096,
//   128 rows 260 -> 176, 256 rows 289 -> 229; 4096 x 14336, 128 rows 52 -> 34,
//   256 rows 65 -> 45, 512 rows 95 -> 69.

#include <torch/all.h>
#include <c10/hip/HIPStream.h>

#include <cmath>

#include "tile_linear.h"
#include "tile_product.h"

namespace vllm_amd {

namespace {

constexpr int TI_ROWS = 256;

// N: columns of out. SILU: w has 2N rows, gate then up; a wave's gate rows,
// then the up rows of the same columns. ONCE: one workgroup reads a weight.
// parts > 1 (not SILU): K is split, and the sums of a part go to `sums` in
// blocks of 32 x 32: [parts][row blocks][column blocks][2][2][lane], those of
// 16 weight rows and in them of 16 rows.
template <typename Tag, bool SILU, bool ONCE, int WGM, int NG, int MG, int PA,
          int PW>
__global__ __launch_bounds__(TP_THREADS, 1) void tile_linear_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const short* __restrict__ w, const int M, const int N, const int K,
    const int m_tiles, const int n_tiles, const int parts,
    f32x4* __restrict__ sums) {
  using P = TileProduct<Tag, WGM, NG, MG, PA, PW>;
  __shared__ __align__(16) char lds[P::LDS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l16 = lane & 15;
  constexpr int H = SILU ? 2 : 1;
  constexpr int NO = P::NI / H;
  const int jobs = m_tiles * n_tiles * parts;
  const int run = (jobs + 7) / 8;
  const int xcd = blockIdx.x % 8, nth = blockIdx.x / 8;
  if (nth >= run || xcd * run + nth >= jobs) return;
  const TileJob t = tile_job(xcd, nth, run, m_tiles, n_tiles);
  const int part = t.part;
  const int m0 = t.m_tile * P::TM;
  const int n0 = t.n_tile * (P::TN / H);
  const int rows = min(M - m0, P::TM);
  const int s0 = tile_part(K / TP_K, part, parts);
  const int steps = tile_part(K / TP_K, part + 1, parts) - s0;
  const short* xt = x + (int64_t)m0 * K;
  const short* wt = w + (int64_t)n0 * K;
  const int turn = t.turn % steps;
  auto stage = [&](int s) {
    s += turn;
    return (s0 + (s >= steps ? s - steps : s)) * TP_K;
  };

  // Byte places of this lane's pieces; rows past the end repeat the last.
  uint32_t ap[P::FA], wp[P::FW];
#pragma unroll
  for (int i = 0; i < P::FA; ++i) {
    const int r = (wave * P::FA + i) * 8 + (lane >> 3);
    ap[i] = (uint32_t)min(r, rows - 1) * (uint32_t)(K * 2) +
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
  P::template run<ONCE>(
      lds, steps, rows,
      [&](int s, int i) { return FillSource{xt + stage(s), ap[i]}; },
      [&](int s, int i) { return FillSource{wt + stage(s), wp[i]}; },
      [&](auto n, auto& acc) {
        constexpr int J = decltype(n)::value;
        const int wm = wave / P::WGN, wn = wave % P::WGN;
        const int col0 = n0 + wn * NO * 16 + row_start16();
        const int cols = n_tiles * (P::TN / 32);
#pragma unroll
        for (int j = 0; j < J; ++j) {
          if (!SILU && parts > 1) {
            const int rb = (m0 + P::row_of(j, wm)) / 32;
            f32x4* to = sums + lane + j % 2 * 64 +
                        (((int64_t)part * m_tiles * (P::TM / 32) + rb) * cols +
                         n0 / 32 + wn * NG) *
                            256;
#pragma unroll
            for (int i = 0; i < P::NI; ++i) to[i * 128] = acc[i][j];
            continue;
          }
          const int row = P::row_of(j, wm) + l16;
          if (row >= rows) continue;
          short* o = out + (int64_t)(m0 + row) * N;
#pragma unroll
          for (int i = 0; i < NO; i += 2) {
            f32x4 v[2] = {acc[i][j], acc[i + 1][j]};
            if constexpr (SILU) {
#pragma unroll
              for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  v[h][r] = v[h][r] / (1.f + __expf(-v[h][r])) *
                            acc[i + h + NO][j][r];
            }
            const i32x4 chunk = row_chunk16<Tag>(v[0], v[1]);
            const int col = col0 + i * 16;
            if (col < N) *reinterpret_cast<i32x4*>(o + col) = chunk;
          }
        }
      });
}

// The parts of a product with K split, added in their order: half a block of
// 32 x 32 a wave, eight parts on their way at once. (The last workgroup of a
// tile to arrive would read all of its parts alone, 7 x 128 KB, at what one CU
// takes in, and the code for it in the kernel above costs its loop registers:
// 4096 x 14336, 256 rows, 8 parts 54.9 us so, 45.2 with this launch.)
template <typename Tag>
__global__ __launch_bounds__(256) void tile_sums_kernel(
    short* __restrict__ out, const f32x4* __restrict__ sums,
    const short* __restrict__ residual, const int M, const int N,
    const int row_blocks, const int col_blocks, const int parts) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int unit = blockIdx.x * 4 + wave;
  const int b = unit % 2, cb = unit / 2 % col_blocks;
  const int rb = unit / 2 / col_blocks;
  if (rb * 32 >= M) return;
  const int64_t part = (int64_t)row_blocks * col_blocks * 256;
  const f32x4* at =
      sums + ((int64_t)rb * col_blocks + cb) * 256 + b * 64 + lane;
  const int row = rb * 32 + b * 16 + (lane & 15);
  s16x4 add[2] = {};
  if (residual != nullptr && row < M) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int col = cb * 32 + c * 16 + (lane >> 4) * 4;
      if (col < N)
        add[c] = *reinterpret_cast<const s16x4*>(residual + (int64_t)row * N +
                                                 col);
    }
  }
  f32x4 v[2];
  constexpr int Q = 8;
  for (int p0 = 0; p0 < parts; p0 += Q) {
    f32x4 t[Q][2];   // (a read past the last part repeats it)
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        t[q][c] = __builtin_nontemporal_load(
            at + min(p0 + q, parts - 1) * part + c * 128);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float a = p0 == 0 ? t[0][c][r] : v[c][r] + t[0][c][r];
#pragma unroll
        for (int q = 1; q < Q; ++q)
          if (p0 + q < parts) a += t[q][c][r];
        v[c][r] = a;
      }
  }
  if (residual != nullptr) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[c][r] += to_f32<Tag>(add[c][r]);
  }
  const i32x4 chunk = row_chunk16<Tag>(v[0], v[1]);
  const int col = cb * 32 + row_start16();
  if (row < M && col < N)
    *reinterpret_cast<i32x4*>(out + (int64_t)row * N + col) = chunk;
}

// us of a product in tiles of `cols` weight rows with K in `parts`, for at most
// 256 workgroups. A stage of 64 columns of K: what a CU takes in, rows of x and
// weights; the weights' way from HBM; products, each by a rate, and between
// their sum and the largest. The rates (a CU's 76 GB/s and 10.8 TFLOP/s, 8 TB/s) are
// coefficients of a fit and not bounds: 1800 times of 33 layers of
// 512 x 7168 to 36864 x 7168 on 72 to 1024 rows are within 7 % of it (rms), and
// the form that it prefers is 0.7 % slower than the best one on average.
double estimate(int64_t M, int64_t N, int64_t K, int cols, int parts) {
  const int64_t tm = M <= 128 ? 128 : 256;
  const int64_t m_tiles = (M + tm - 1) / tm;
  const double jobs = (double)(m_tiles * ((N + cols - 1) / cols) * parts);
  const double rows = (double)(m_tiles == 1 ? (M + 31) / 32 * 32 : tm);
  auto pow = [](double v) { return std::pow(v, 1.85); };
  const double stage =
      std::pow(pow((rows + cols) * 0.128 / 76.) +
                   pow(cols * 128e-6 * jobs / (double)m_tiles / 8.) +
                   pow(rows * cols * 128e-6 / 10.8),
               1 / 1.85);
  return (double)K / TP_K / parts * stage + 5.4 +
         (parts > 1 ? 3.5 + parts * (double)M * (double)N * 4e-6 / 3.2 : 0.);
}

// The form of least estimate among those of one round that keep enough of the
// CUs busy, where it is ahead of the library.
//
// With K split (up to 16 parts) 60 % are enough. From K = 5120 on up to 128
// rows, above from 6144 on, and only if K is long beside the 256 x 256 tiles of
// the output (170 columns of K each, 90 of them), since partial sums cost 10 to
// 20 us. Below 1536 columns of output there is too little to split. us, the
// library and this (at 128, 256 and 1024 rows if not said): 4096 x 14336 52 /
// 34, 65 / 45, 137 / 116; 3584 x 18944 65 / 40, 80 / 52, 173 / 132; 7168 x
// 16384 71 / 54, 107 / 72, and 512 rows 148 / 117; 2112 x 7168 25 / 17, 32 /
// 24, 49 / 45. On the other side of the lines: 4096 x 4096 17.3 / 17.0, 21.0 /
// 25.1, 41 / 50; 4096 x 7168, 1024 rows 69 / 74; 8192 x 28672, 768 rows 301 /
// 316; 512 x 7168, 256 rows 12 / 15.6. Of 2300 sizes inside 0.74 of the
// library's time on average, one above 1.02 (1.026).
//
// With K whole, up to 256 rows: 65 %, and 75 % where K is long (the library
// begins K at several places: 19712 x 9728, 148 rows, 60 % busy 105 / 113;
// 39680 x 10240, 68 rows, 61 % 157 / 169; 22272 x 5632, 95 rows, 68 % 57 / 61;
// 43456 x 11968, 154 rows, 66 % 216 / 229; inside 22016 x 4096, 192 rows, 67 %
// 62 / 52). Tiles of 64 take x in for few weights: up to 128 rows 60 % are
// enough (24576 x 1536 27.6 / 23.0), above only nearly all, and K up to 5120
// (256 rows: 16384 x 4096 52 / 48, 71 % 11568 x 4096 39 / 45, 88 % 14336 x 4096
// 45 / 47; 15872 x 7168 78 / 82). Of 1200 sizes inside 0.87 on average, two
// above 1.03 (1.05).
TileForm by_estimate(int64_t M, int64_t N, int64_t K) {
  TileForm best{0, 1};
  if (M > 1024) return best;
  const int64_t tm = M <= 128 ? 128 : 256;
  const int64_t out_tiles = (M + 255) / 256 * ((N + 255) / 256);
  const bool split = N >= 1536 && (M <= 128 ? K >= 5120
                                            : K >= 6144 && out_tiles <= 90 &&
                                                  K >= 170 * out_tiles);
  double least = 1e30;
  for (int cols : {64, 128, 256}) {
    if (cols == 64 && M > 256) continue;
    const int64_t tiles = (M + tm - 1) / tm * ((N + cols - 1) / cols);
    const int64_t lengthy = cols == 256 ? 8192 : M <= 128 ? 5120 : 7168;
    const int64_t whole = cols > 64 ? (K > lengthy ? 192 : 167)
                          : M <= 128 ? 154 : K <= 5120 ? 241 : 257;
    for (int parts = 1; parts <= 16 && tiles * parts <= 256; ++parts) {
      if (tiles * parts < (parts == 1 ? whole : 154) ||
          K / TP_K / parts < 4 ||
          (parts == 1 ? M > 256 || M <= 64 || K <= 8 * M : !split))
        continue;
      const double t = estimate(M, N, K, cols, parts);
      if (t < least) {
        least = t;
        best = {cols, parts};
      }
    }
  }
  return best;
}

// How M rows meet rows_w weight rows of K; cols 0: in the library, or up to 64
// rows in stream_linear.hip.
//
// On 33 to 64 rows stream_linear splits K over the waves of a workgroup, which
// takes x in for 16 to 128 weight rows; a tile takes it in for 128 or 256. So
// tiles are ahead where their rounds keep the CUs busy, the more the shorter K
// is, and where K is long enough to be split here: from 10400 on 33 rows (the
// crossing lies between 8700 and 11000 by the weight rows) to 8400 on 64 (6600
// to 8700), later where there are few weight rows, whose parts are many. us,
// stream_linear and this, 64 rows: 128256 x 4096 190 and 172; 57344 x 4096 90
// and 75; 102400 x 2048 (0.78 of two rounds) 96 and 80, 152064 x 3584 216 and
// 207; 57344 x 8192 with the activation 159 and 146; 28672 x 4096 with it 41.9
// and 40.9; on 33 and 64 rows 5120 x 10240 27.3 and 24.8, 29.7 and 25.9; 3072 x
// 12288 23.0 and 21.6, 25.5 and 22.4; 8192 x 10240 35.1 and 33.5, 38.5 and
// 34.7; 7168 x 16384 on 64 52.9 and 45.0, 8192 x 28672 103 and 83. On the other
// side: 145000 x 5504 by tiles of 128 311 and 330; 24576 x 1536 18.1 and 18.7;
// 12288 x 5120 29.5 and 31.0; 8192 x 8192 on 33 and 64 27.9 and 31.1, 29.7 and
// 31.1; 5120 x 8192 on 33 21.8 and 22.0; 2560 x 10752 on 48 4 % behind; 22880 x
// 12096 on 40 13 % (two parts). Where all CUs take gate and up rows at a stride
// of 8 KB they meet on few channels: 32768 x 4096 with the activation 43.3 and
// 50.4, 31600 x 4096 42.6 and 42.0. 8100 sizes inside: 0.90 of stream_linear's
// time on average, one in 180 above 1.02, seven above 1.05 (1.074: 7168 x 13312
// on 33).
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
TileForm tile_form(int64_t M, int64_t rows_w, int64_t K, bool silu) {
  if (M <= 32 || (silu && M > TI_ROWS)) return {0, 1};
  auto rounds = [&](int tile) {
    return (rows_w + tile * 256 - 1) / tile / 256;
  };
  auto busy = [&](int tile) {
    return (double)((rows_w + tile - 1) / tile) / (double)(rounds(tile) * 256);
  };
  if (M <= 64) {
    if (K < 2048) return {0, 1};
    if (busy(256) >= (rounds(256) == 1 ? 0.85
                      : K > 4096       ? 0.9
                      : silu           ? 0.76
                                       : 0.75))
      return {256, 1};
    const bool meet = silu && K % 4096 == 0 && busy(128) > 0.97;
    if (K <= 5120 && busy(128) >= 0.85 && !meet) return {128, 1};
    if (silu || rows_w < 2304 || rows_w > 19456 ||
        K < 12500 - 64 * M + (rows_w < 2816 ? 4000 : 0))
      return {0, 1};
  } else if (M <= TI_ROWS && (silu || K > 8 * M)) {
    if (busy(256) >= 0.95 && (silu || M > 128 || rounds(256) > 1))
      return {256, 1};
    const double least =
        rounds(128) > 1 ? (silu ? 0.9 : 2.) : silu ? 0.65 : 0.95;
    if (busy(128) >= least) return {128, 1};
  }
  return silu ? TileForm{0, 1} : by_estimate(M, rows_w, K);
}

template <typename Tag, bool SILU>
void launch(torch::Tensor& out, const torch::Tensor& x,
            const torch::Tensor& w, TileForm form,
            const short* residual = nullptr) {
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)out.size(1);
  constexpr int H = SILU ? 2 : 1;
  const int tm = M <= 128 ? 128 : 256;
  const int m_tiles = ceil_div(M, tm), n_tiles = ceil_div(N, form.cols / H);
  const int jobs = m_tiles * n_tiles * form.parts;
  const int row_blocks = m_tiles * (tm / 32);
  const int col_blocks = n_tiles * (form.cols / 32);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  torch::Tensor sums;
  if (form.parts > 1)
    sums = torch::empty({(int64_t)form.parts * row_blocks * col_blocks * 1024},
                        x.options().dtype(torch::kFloat));
  f32x4* const to = form.parts > 1 ? (f32x4*)sums.data_ptr() : nullptr;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(ceil_div(jobs, 8) * 8), dim3(TP_THREADS),
                       0, stream, (short*)out.data_ptr(),
                       (const short*)x.data_ptr(), (const short*)w.data_ptr(),
                       M, N, K, m_tiles, n_tiles, form.parts, to);
  };
  if (M <= 128) {
    if (form.cols == 128)
      go(tile_linear_kernel<Tag, SILU, true, 2, 2, 2, 5, 5>);
    else if (form.cols == 256)
      go(tile_linear_kernel<Tag, SILU, true, 1, 2, 4, 3, 3>);
    else if constexpr (!SILU)
      go(tile_linear_kernel<Tag, SILU, true, 4, 2, 1, 5, 5>);
  } else if (m_tiles == 1) {
    if (form.cols == 128)
      go(tile_linear_kernel<Tag, SILU, true, 2, 2, 4, 3, 3>);
    else if (form.cols == 256)
      go(tile_linear_kernel<Tag, SILU, true, 2, 4, 4, 2, 3>);
    else if constexpr (!SILU)
      go(tile_linear_kernel<Tag, SILU, true, 4, 2, 2, 3, 3>);
  } else if constexpr (!SILU) {
    if (form.cols == 128)
      go(tile_linear_kernel<Tag, SILU, false, 2, 2, 4, 3, 3>);
    else
      go(tile_linear_kernel<Tag, SILU, false, 2, 4, 4, 2, 3>);
  }
  if (form.parts > 1)
    hipLaunchKernelGGL((tile_sums_kernel<Tag>),
                       dim3(ceil_div(row_blocks * col_blocks * 2, 4)),
                       dim3(256), 0, stream, (short*)out.data_ptr(), to,
                       residual, M, N, row_blocks, col_blocks, form.parts);
}

}  // namespace

// The form for a product of these sizes, 0 if it is not one for this file.
TileForm tile_linear_form(int64_t M, int64_t rows_w, int64_t K, bool silu) {
  if (rows_w <= 0 || rows_w % (silu ? 16 : 8) != 0 || K <= 0 ||
      K % TP_K != 0 || K >= (1 << 22) || (rows_w + 256) * K * 2 >= (1ll << 32))
    return {0, 1};
  return tile_form(M, rows_w, K, silu);
}

// For the tests: {XCD, part of K, row tile, weight tile, first stage in the
// part} of every workgroup of a product of these sizes; nothing if it is not
// one for this file.
std::vector<int64_t> linear_starts(int64_t rows, int64_t weight_rows,
                                   int64_t k, bool silu) {
  const TileForm form = tile_linear_form(rows, weight_rows, k, silu);
  std::vector<int64_t> out;
  if (form.cols == 0) return out;
  const int m_tiles = ceil_div((int)rows, rows <= 128 ? 128 : 256);
  const int n_tiles = ceil_div((int)weight_rows, form.cols);
  const int jobs = m_tiles * n_tiles * form.parts;
  const int run = ceil_div(jobs, 8), stages = (int)k / TP_K;
  for (int xcd = 0; xcd < 8; ++xcd)
    for (int nth = 0; nth < run && xcd * run + nth < jobs; ++nth) {
      const TileJob t = tile_job(xcd, nth, run, m_tiles, n_tiles);
      const int steps = tile_part(stages, t.part + 1, form.parts) -
                        tile_part(stages, t.part, form.parts);
      out.insert(out.end(), {xcd, t.part, t.m_tile, t.n_tile, t.turn % steps});
    }
  return out;
}

// The product of x [M, K] and w [rows, K], both contiguous, into out [M, n],
// if it is one that this file takes. With a residual [M, n] (8 B places, not
// beside an activation) the sum of both, if K is split: it is added with the
// parts then.
bool tile_linear_add(torch::Tensor& out, const torch::Tensor& x,
                     const torch::Tensor& w, bool silu,
                     const short* residual) {
  const int64_t K = x.size(1);
  const TileForm form = tile_linear_form(x.size(0), w.size(0), K, silu);
  if (form.cols == 0 ||
      (residual != nullptr && (silu || form.parts == 1)) || w.size(1) != K ||
      w.scalar_type() != x.scalar_type() ||
      (x.scalar_type() != torch::kBFloat16 &&
       x.scalar_type() != torch::kHalf) ||
      !x.is_contiguous() || !w.is_contiguous() ||
      (uintptr_t)x.data_ptr() % 16 != 0 || (uintptr_t)w.data_ptr() % 16 != 0)
    return false;
  if (x.scalar_type() == torch::kBFloat16) {
    if (silu) launch<BF16Tag, true>(out, x, w, form);
    else      launch<BF16Tag, false>(out, x, w, form, residual);
  } else {
    if (silu) launch<FP16Tag, true>(out, x, w, form);
    else      launch<FP16Tag, false>(out, x, w, form, residual);
  }
  HIP_CHECK_KERNEL();
  return true;
}

bool tile_linear(torch::Tensor& out, const torch::Tensor& x,
                 const torch::Tensor& w, bool silu) {
  return tile_linear_add(out, x, w, silu, nullptr);
}

}  // namespace vllm_amd
