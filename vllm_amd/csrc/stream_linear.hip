// Linear layers on few rows for MI355X (gfx950):
//   out[M, N] = x[M, K] @ w[N, K]^T (+ bias), 16-bit operands, fp32 sums,
// and the same with silu(gate) * up of two halves of w as the epilogue.
//
// Up to 64 rows every weight is used too little for anything but HBM to
// bound the product, if the weights keep coming. Three things decide that:
//
//  * Whole 128 B lines. A wave that loads fragments directly takes 64 B of
//    16 rows at a time; each half line costs as much as a whole one on the
//    way from L2, and rows of x, read again by every workgroup, run into
//    that first (4096 x 4096, us for 1 / 8 / 64 rows: fragments directly
//    8.1 / 9.5 / 23.9, through LDS in whole lines 8.1 / 8.4 / 13.1).
//  * No waiting on other waves. A wave takes every WV-th run of 64 columns
//    of K for all rows of its workgroup's tile, so it fills its own ring in
//    LDS (8 rows x 128 B an instruction, no registers) and waits for its own
//    fills only; sums meet once, at the end. Each line enters a workgroup
//    once. Workgroups begin at different places of K, so that they do not
//    all ask for the same lines of x at a time (28672 x 4096, 64 rows: 48.8
//    -> 45.7 us).
//  * Enough workgroups of equal size (plan() below). Narrow layers split K
//    over workgroups; the last one to arrive adds up the parts in their
//    order (arrivals.h; 2112 x 7168, 64 rows: 14.3 us in three parts, 21.3
//    in one).
//  * Weights leave L2 first (lds_fill16_once): read once, they would push
//    out x, which every workgroup reads (7168 x 16384, 64 rows 58 -> 49 us).
//
// us on weights from HBM, tuned library products -> these, in a graph (in
// brackets the weights' bytes at 6.6 TB/s, which streams of this kind reach on
// average; the widest layer passes it):
//                   1 row          8 rows         32 rows        64 rows
//    4096 x 4096    10.4 ->  7.5   13.4 ->  7.6   11.7 ->  9.8   14.0 -> 12.4   (5.1)
//    6144 x 4096    15.2 -> 11.1   14.2 -> 11.3   14.9 -> 14.8   18.2 -> 17.7   (7.6)
//   28672 x 4096    48.9 -> 37.3   52.1 -> 37.4   52.4 -> 38.8   53.9 -> 42.9   (36)
//    4096 x 14336   25.3 -> 20.3   25.4 -> 21.2   31.6 -> 25.0   37.5 -> 28.7   (18)
//    2112 x 7168    12.2 ->  8.3   12.4 ->  9.8   16.0 -> 11.1   19.2 -> 14.3   (4.6)
//  128256 x 4096     175 ->  154    174 ->  151    188 ->  163    199 ->  186   (159)
// (From 33 rows on tile_linear.hip takes the third, the fourth and the last
// without a bias: 42, 28 and 172 on 64.)

#include <torch/all.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cmath>

#include "arrivals.h"
#include "stream_product.h"
#include "tile_linear.h"

namespace vllm_amd {

// gemm_hipblaslt.cpp, elementwise.hip
torch::Tensor lt_linear(torch::Tensor a, torch::Tensor w,
                        c10::optional<torch::Tensor> bias);
torch::Tensor silu_and_mul(torch::Tensor x);
// tile_linear.hip
bool tile_linear(torch::Tensor& out, const torch::Tensor& x,
                 const torch::Tensor& w, bool silu);

namespace {

constexpr int SL_ROWS = 64;      // rows of x at most
constexpr int SL_PARTS = 8;      // of K, over workgroups
constexpr int SL_JOBS = 1024;    // column tiles whose K is split
constexpr int SL_LDS = 160 * 1024;

// Forms: 16-row groups of w per workgroup, waves, ring steps per wave.
struct Form { int ni, wv, d; };
constexpr Form SL_FORMS[] = {{1, 8, 4}, {2, 4, 2}, {4, 4, 2},
                             {6, 4, 2}, {8, 4, 2}, {8, 2, 2},
                             {10, 2, 2}};
constexpr int SL_NFORMS = sizeof(SL_FORMS) / sizeof(Form);

// Groups of 8 rows of x that a launch for M rows is made for.
constexpr int row_groups(int64_t M) {
  return M <= 8 ? 1 : M <= 16 ? 2 : M <= 32 ? 4 : 8;
}

// xg: groups of 8 rows of x.
constexpr int ring_bytes(Form f, int xg) {
  return f.wv * f.d * (2 * f.ni + xg) * SP_FILL;
}
constexpr int sums_bytes(Form f, int xg) {
  return f.wv * f.ni * ((xg + 1) / 2) * WAVE_SIZE * 16;
}
constexpr int lds_bytes(Form f, int xg) {
  return ring_bytes(f, xg) > sums_bytes(f, xg) ? ring_bytes(f, xg)
                                               : sums_bytes(f, xg);
}

// N: columns of out. SILU: w has 2N rows, gate then up; a tile is NI / 2
// groups of gate rows and the NI / 2 groups of the same columns' up rows.
template <typename Tag, int NI, int XG, int WV, int D, bool SILU>
__global__ __launch_bounds__(WV * WAVE_SIZE) void stream_linear_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const short* __restrict__ w, const short* __restrict__ bias, const int M,
    const int N, const int K, const int n_tiles, const int parts,
    f32x4* __restrict__ part_sums, unsigned* __restrict__ arrived) {
  using P = StreamProduct<Tag, NI, XG, WV, D>;
  constexpr int MT = P::MT;
  constexpr int NO = SILU ? NI / 2 : NI;
  extern __shared__ __align__(16) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  const int tile = blockIdx.x % n_tiles;
  const int part = blockIdx.x / n_tiles;
  const int n0 = tile * NO * 16;

  // Rows past the end repeat the last.
  uint32_t wat[2 * NI], xat[XG];
#pragma unroll
  for (int i = 0; i < 2 * NI; ++i) {
    const int r = i * 8 + (lane >> 3);
    const int half = SILU && i >= NI ? 1 : 0;
    wat[i] = sp_place(min(r - half * NO * 16, N - 1 - n0) + half * N, r, K);
  }
#pragma unroll
  for (int i = 0; i < XG; ++i) {
    const int r = i * 8 + (lane >> 3);
    xat[i] = sp_place(min(r, M - 1), r, K);
  }
  const int steps = K / SP_K;
  P::run(lds, wave, steps * part / parts, steps * (part + 1) / parts,
         blockIdx.x / 8, reinterpret_cast<const char*>(w + (int64_t)n0 * K),
         wat, reinterpret_cast<const char*>(x), xat);

  // Each wave goes on with a share of the tiles.
  constexpr int T = P::T;
  constexpr int TO = NO * MT;
  constexpr int PER = (TO + WV - 1) / WV;
  constexpr int H = SILU ? 2 : 1;
  f32x4 v[PER][H];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = u * WV + wave;
    if (t >= TO) break;
#pragma unroll
    for (int h = 0; h < H; ++h) v[u][h] = P::sum(lds, h * TO + t);
  }
  if (parts > 1) {
    f32x4* sums = part_sums + (int64_t)tile * parts * T * WAVE_SIZE + lane;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int t = u * WV + wave;
      if (t >= TO) break;
#pragma unroll
      for (int h = 0; h < H; ++h)
        part_put(sums + (part * T + h * TO + t) * WAVE_SIZE, v[u][h]);
    }
    if (!last_to_arrive(arrived, tile, parts,
                        reinterpret_cast<unsigned*>(lds)))
      return;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int t = u * WV + wave;
      if (t >= TO) break;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        // On their way at once, added in their order (a read past the last
        // part repeats it: with a branch each read waits for the one before).
        const f32x4* at = sums + (h * TO + t) * WAVE_SIZE;
        auto add = [&](auto n) {
          constexpr int Q = decltype(n)::value;
          f32x4 p[Q];
#pragma unroll
          for (int q = 0; q < Q; ++q)
            p[q] = part_get(at + min(q, parts - 1) * (T * WAVE_SIZE));
          v[u][h] = p[0];
#pragma unroll
          for (int q = 1; q < Q; ++q)
            if (q < parts) v[u][h] += p[q];
        };
        if (parts == 2)     add(std::integral_constant<int, 2>{});
        else if (parts < 5) add(std::integral_constant<int, 4>{});
        else                add(std::integral_constant<int, SL_PARTS>{});
      }
    }
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = u * WV + wave;
    if (t >= TO) break;
    const int row = (t % MT) * 16 + l16;
    const int col = n0 + (t / MT) * 16 + l4 * 4;
    f32x4 o = v[u][0];
    if constexpr (SILU) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[r] = o[r] / (1.f + __expf(-o[r])) * v[u][1][r];
    }
    if (row >= M || col >= N || (XG == 1 && l16 >= 8)) continue;
    if (!SILU && bias != nullptr) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] += to_f32<Tag>(bias[col + r]);
    }
    *reinterpret_cast<int2*>(out + (int64_t)row * N + col) =
        int2{pack2<Tag>(o[0], o[1]), pack2<Tag>(o[2], o[3])};
  }
}

struct Plan { int form, parts; };

// Form and parts of K by an estimate of the time. Its terms (added as fourth
// powers): weights at 6 TB/s; all that enters workgroups, x again in each, at
// 15 TB/s; what the fullest CU takes in at 60 GB/s, evened out by two fifths
// where neighbours still run. A workgroup's start costs 0.2 us of its CU,
// splitting K 1.5 us and the traffic of partial sums. These are coefficients
// of a fit and not bounds (the first is passed by a tenth): they come closest
// to the best of all forms over 15 layers of 2112 x 7168 to 128256 x 4096 at 1
// to 64 rows, 1.3 % from it on average, 7 % at most.
Plan plan(int xg, int64_t rows_w, int K, bool silu) {
  Plan best{-1, 1};
  double least = 1e30;
  auto fourth = [](double v) { return v * v * v * v; };
  for (int i = 0; i < SL_NFORMS; ++i) {
    const Form f = SL_FORMS[i];
    // Two waves have too little on the way where four fit.
    if (lds_bytes(f, xg) > SL_LDS || (f.wv == 2 && xg < 8) ||
        (silu && f.ni % 2 != 0))
      continue;
    const int64_t tiles = (rows_w + f.ni * 16 - 1) / (f.ni * 16);
    for (int parts : {1, 2, 3, 4, 6, 8}) {
      if (parts > 1 && (tiles > SL_JOBS || tiles * parts > 1100 ||
                        K / SP_K / parts < f.wv))
        continue;
      const double mb = (f.ni * 16 + xg * 8) * 2e-6 * K / parts;
      const double jobs = (double)(tiles * parts);
      const double cus = (double)((tiles * parts + 255) / 256);
      const double load =
          cus > 1 && lds_bytes(f, xg) * 2 > SL_LDS
              ? cus
              : 0.6 * cus + 0.4 * std::max(1.0, jobs / 256);
      double t = std::sqrt(std::sqrt(fourth(rows_w * 2e-6 * K / 6.0) +
                                     fourth(jobs * mb / 15.0) +
                                     fourth(load * mb / 0.06))) +
                 0.2 * jobs / 256;
      if (parts > 1) t += 1.5 + 0.04 * parts * f.ni * xg;
      if (t < least) {
        least = t;
        best = {i, parts};
      }
    }
  }
  return best;
}

template <typename Tag, int I, int XG, bool SILU>
void launch_form(torch::Tensor& out, const torch::Tensor& x,
                 const torch::Tensor& w, const short* bias, int N,
                 int parts) {
  constexpr Form f = SL_FORMS[I];
  if constexpr (lds_bytes(f, XG) <= SL_LDS && (f.wv > 2 || XG == 8) &&
                (!SILU || f.ni % 2 == 0)) {
    const int M = (int)x.size(0), K = (int)x.size(1);
    const int cols = f.ni * 16 / (SILU ? 2 : 1);
    const int tiles = ceil_div(N, cols);
    torch::Tensor sums, arrived;
    if (parts > 1) {
      sums = torch::empty({(int64_t)tiles * parts * f.ni * ((XG + 1) / 2) *
                           WAVE_SIZE * 4},
                          x.options().dtype(torch::kFloat));
      arrived = arrival_counters(x, tiles);
    }
    hipLaunchKernelGGL(
        (stream_linear_kernel<Tag, f.ni, XG, f.wv, f.d, SILU>),
        dim3(tiles * parts), dim3(f.wv * WAVE_SIZE), lds_bytes(f, XG),
        c10::hip::getCurrentHIPStream().stream(), (short*)out.data_ptr(),
        (const short*)x.data_ptr(), (const short*)w.data_ptr(), bias, M, N, K,
        tiles, parts, parts > 1 ? (f32x4*)sums.data_ptr() : nullptr,
        parts > 1 ? (unsigned*)arrived.data_ptr() : nullptr);
  } else {
    TORCH_CHECK(false, "stream_linear: form does not fit");
  }
}

template <typename Tag, bool SILU>
void launch(torch::Tensor& out, const torch::Tensor& x,
            const torch::Tensor& w, const short* bias, int N) {
  const int xg = row_groups(x.size(0));
  const Plan p = plan(xg, w.size(0), (int)x.size(1), SILU);
  auto by_rows = [&](auto form) {
    constexpr int I = decltype(form)::value;
    if (xg == 1) launch_form<Tag, I, 1, SILU>(out, x, w, bias, N, p.parts);
    else if (xg == 2) launch_form<Tag, I, 2, SILU>(out, x, w, bias, N, p.parts);
    else if (xg == 4) launch_form<Tag, I, 4, SILU>(out, x, w, bias, N, p.parts);
    else launch_form<Tag, I, 8, SILU>(out, x, w, bias, N, p.parts);
  };
  static_assert(SL_NFORMS == 7);
  switch (p.form) {
    case 0: return by_rows(std::integral_constant<int, 0>{});
    case 1: return by_rows(std::integral_constant<int, 1>{});
    case 2: return by_rows(std::integral_constant<int, 2>{});
    case 3: return by_rows(std::integral_constant<int, 3>{});
    case 4: return by_rows(std::integral_constant<int, 4>{});
    case 5: return by_rows(std::integral_constant<int, 5>{});
    case 6: return by_rows(std::integral_constant<int, 6>{});
    default: TORCH_CHECK(false, "stream_linear: no form");
  }
}

}  // namespace

// Whether a product of M rows with rows_w weight rows (silu: n = rows_w / 2
// columns of out) is one for this file, by its sizes. Up to 64 rows it is,
// but for two kinds at which the tuned library is ahead (and callers ask
// tile_linear_first before):
//  * Wide and short ones. Workgroups hardly begin before they end, and what
//    they write is no longer little beside the weights. us, library and this:
//    50272 x 768, 16 / 32 / 64 rows 18.4 and 18.9, 19.1 and 20.5, 20.5 and
//    26.9, x 2048 40 and 36 (64 rows); 65536 x 256, 8 / 32 / 64 rows 9.8 and
//    10.8, 12.5 and 13.0, 11.7 and 17.7; 32000 x 512, 32 / 64 rows 10.7 and
//    9.5, 10.9 and 12.2. An activation as epilogue makes up for most of it
//    (131072 x 512, 64 rows 49 and 51).
//  * Narrow ones of more than 32 rows: a few workgroups take in all of x (128
//    x 7168, 32 / 64 rows 8.4 and 7.2, 8.4 and 9.5; 512 x 7168, 64 rows 10.8
//    and 9.8; 128 x 14336 12.9 and 11.4; where K is shorter the library takes
//    5.2 to 12.7, by the algorithm that its race came to).
bool stream_sizes(int64_t M, int64_t rows_w, int64_t n, int64_t K) {
  if (M <= 0 || M > SL_ROWS || n <= 0 || n % 4 != 0 || K <= 0 ||
      K % SP_K != 0 || K >= (1 << 24) || rows_w >= (1 << 30) ||
      (rows_w + 160) * K * 2 >= (1ll << 32))
    return false;
  if (rows_w != n) return !(M > 32 && n >= 49152 && K <= 1024);
  if (rows_w >= 49152 && K <= std::min(256 * row_groups(M), 1536))
    return false;
  if (M > 32 && rows_w >= 24576 && K <= 1024) return false;
  return !(M > 32 && rows_w <= 256 && K >= 6144 && K <= 8192);
}

// Whether stream_linear takes the product: x [M, K] and w [rows, K], both
// contiguous; out has n columns.
bool stream_linear_takes(const torch::Tensor& x, const torch::Tensor& w,
                         int64_t n) {
  return stream_sizes(x.size(0), w.size(0), n, x.size(1)) &&
         (x.scalar_type() == torch::kBFloat16 ||
          x.scalar_type() == torch::kHalf) &&
         w.scalar_type() == x.scalar_type() && w.size(1) == x.size(1) &&
         x.is_contiguous() && w.is_contiguous() &&
         (uintptr_t)x.data_ptr() % 16 == 0 &&
         (uintptr_t)w.data_ptr() % 16 == 0;
}

// What a product of these sizes runs as, for 16-bit operands that begin on
// 16 B: {0} the library, {1, 16-row groups of weights, waves, ring steps,
// 8-row groups of x, parts of K} stream_linear, {2, weight rows of a tile,
// parts of K} tile_linear.
std::vector<int64_t> linear_form(int64_t rows, int64_t weight_rows, int64_t k,
                                 bool silu) {
  const int64_t n = silu ? weight_rows / 2 : weight_rows;
  if (!tile_linear_first(rows, weight_rows, k, silu) &&
      stream_sizes(rows, weight_rows, n, k)) {
    const int xg = row_groups(rows);
    const Plan p = plan(xg, weight_rows, (int)k, silu);
    const Form f = SL_FORMS[p.form];
    return {1, f.ni, f.wv, f.d, xg, p.parts};
  }
  const TileForm tile = tile_linear_form(rows, weight_rows, k, silu);
  if (tile.cols == 0) return {0};
  return {2, tile.cols, tile.parts};
}

// x, w and bias as stream_linear_takes and lt_linear have checked them.
torch::Tensor stream_linear(const torch::Tensor& x, const torch::Tensor& w,
                            const c10::optional<torch::Tensor>& bias) {
  const int64_t N = w.size(0);
  auto out = torch::empty({x.size(0), N}, x.options());
  const short* b = bias.has_value() ? (const short*)bias->data_ptr() : nullptr;
  if (x.scalar_type() == torch::kBFloat16)
    launch<BF16Tag, false>(out, x, w, b, (int)N);
  else
    launch<FP16Tag, false>(out, x, w, b, (int)N);
  HIP_CHECK_KERNEL();
  return out;
}

// silu(x @ gate^T) * (x @ up^T), w = [gate; up]; in one launch where this file
// or tile_linear takes it (the products are then not rounded in between).
torch::Tensor linear_silu_and_mul(torch::Tensor a, torch::Tensor w) {
  TORCH_CHECK(w.dim() == 2 && w.size(0) % 2 == 0 && a.dim() >= 1 &&
              a.size(-1) == w.size(1) && a.scalar_type() == w.scalar_type(),
              "linear_silu_and_mul: [.., K] x [2N, K]");
  auto sizes = a.sizes().vec();
  auto x = a.reshape({-1, sizes.back()}).contiguous();
  const int64_t N = w.size(0) / 2;
  sizes.back() = N;
  auto out = torch::empty({x.size(0), N}, x.options());
  if (tile_linear_first(x.size(0), w.size(0), x.size(1), true) ||
      !stream_linear_takes(x, w, N)) {
    if (x.size(0) > 0 && tile_linear(out, x, w, true))
      return out.reshape(sizes);
    return silu_and_mul(lt_linear(x, w, c10::nullopt)).reshape(sizes);
  }
  if (x.scalar_type() == torch::kBFloat16)
    launch<BF16Tag, true>(out, x, w, nullptr, (int)N);
  else
    launch<FP16Tag, true>(out, x, w, nullptr, (int)N);
  HIP_CHECK_KERNEL();
  return out.reshape(sizes);
}

}  // namespace vllm_amd
