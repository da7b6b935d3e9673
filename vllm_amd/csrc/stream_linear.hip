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
#include <initializer_list>

#include "arrivals.h"
#include "stream_product.h"
#include "tile_linear.h"

namespace vllm_amd {

// gemm_hipblaslt.cpp, elementwise.hip, pooled_attention.hip
torch::Tensor lt_linear(torch::Tensor a, torch::Tensor w,
                        c10::optional<torch::Tensor> bias);
torch::Tensor silu_and_mul(torch::Tensor x);
torch::Tensor silu_and_mul_any(torch::Tensor x);
torch::Tensor rms_norm(torch::Tensor x, torch::Tensor weight, double eps);
torch::Tensor linear_silu_and_mul(torch::Tensor a, torch::Tensor w);
void rope_and_cache(torch::Tensor positions, torch::Tensor q, torch::Tensor k,
                    torch::Tensor v, torch::Tensor cos_sin_cache, int64_t rot,
                    torch::Tensor kv_cache, torch::Tensor slot_mapping);
// tile_linear.hip
bool tile_linear(torch::Tensor& out, const torch::Tensor& x,
                 const torch::Tensor& w, bool silu);
bool tile_linear_add(torch::Tensor& out, const torch::Tensor& x,
                     const torch::Tensor& w, bool silu, const short* residual);

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
constexpr int sums_bytes(Form f, int xg, bool norm) {
  return f.wv * (f.ni * ((xg + 1) / 2) + norm) * WAVE_SIZE * 16;
}
// norm_steps: steps of K of a workgroup that takes gains, else 0.
constexpr int lds_bytes(Form f, int xg, int norm_steps = 0) {
  const int sums = sums_bytes(f, xg, norm_steps > 0);
  return (ring_bytes(f, xg) > sums ? ring_bytes(f, xg) : sums) +
         (norm_steps > 0 ? f.wv * sp_gain_bytes(norm_steps, f.wv) : 0);
}

// What a product has beside its operands, all of it optional.
struct Beside {
  const short* bias = nullptr;       // [N]
  const short* residual = nullptr;   // [M, N], added to the result
  const short* gains = nullptr;      // [K], of the RMS norm of x
  float eps = 0.f;
};

// What becomes of two halves of weight rows: nothing (one row a column),
// silu(gate) * up, or the rotation of a head's halves.
enum { SINGLE = 0, SILU = 1, ROPE = 2 };

// Weights of query, key and value heads. out gets the rotated queries [M,
// q_heads, 2 * half], the cache [2, blocks, kv_heads, block_size, 2 * half] the
// rotated keys and the values.
struct Heads {
  const int64_t* positions = nullptr;   // [M]
  const int64_t* slots = nullptr;       // [M]
  const float* cos_sin = nullptr;       // [positions, cos half | sin half]
  void* kv_cache = nullptr;
  int64_t plane = 0;                    // elements from keys to values
  int half = 0, q_heads = 0, kv_heads = 0, block_size = 0;
  bool fp8 = false;
};

// N: columns of out. PAIR SILU: w has 2N rows, gate then up; a tile is NI / 2
// groups of gate rows and the NI / 2 groups of the same columns' up rows. ROPE:
// N counts pairs of a head's columns that turn together, and a tile is NI / 2
// groups of first and of second ones of one head. (The launch for rotation and
// cache took 2.9 us of a layer: the same, 1 row 508 -> 498 us, 8 rows 512 ->
// 502. What it read is asked for behind the first fills here, as the residual
// is, or it would be waited for at the end.)
// NORM: the product of x's RMS norm. A row's root comes out of the sum, so a
// workgroup needs its squares at the end only, and has them, since all of x
// passes through it. What meets the weights is x * gain instead of x * root *
// gain, rounded once to the same bits. Where a row lies between powers of two
// is another place then, so the rounding's share of the result is 0.93 to 1.05
// of what it was, by the rows' size. With the residual as epilogue a layer of
// few rows keeps no launch for its norms: they took 3.5 us each beside products
// of 7 to 37 (four layers of 4096 and the logits, 1 row 526 -> 508 us, 8 rows 534
// -> 512).
template <typename Tag, int NI, int XG, int WV, int D, int PAIR, bool NORM>
__global__ __launch_bounds__(WV * WAVE_SIZE) void stream_linear_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const short* __restrict__ w, const Beside beside, const Heads heads,
    const int M, const int N, const int K, const int n_tiles, const int parts,
    f32x4* __restrict__ part_sums, unsigned* __restrict__ arrived) {
  using P = StreamProduct<Tag, NI, XG, WV, D, NORM>;
  constexpr int MT = P::MT;
  constexpr int NO = PAIR ? NI / 2 : NI;
  extern __shared__ __align__(16) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  const int tile = blockIdx.x % n_tiles;
  const int part = blockIdx.x / n_tiles;
  const int n0 = tile * NO * 16;
  // Weight row of column n0, and how far the other half's lies.
  const int head = PAIR == ROPE ? n0 / heads.half : 0;
  const int w0 = n0 + head * heads.half;
  const int apart = PAIR == ROPE ? heads.half : N;

  // Rows past the end repeat the last.
  uint32_t wat[2 * NI], xat[XG];
#pragma unroll
  for (int i = 0; i < 2 * NI; ++i) {
    const int r = i * 8 + (lane >> 3);
    const int half = PAIR && i >= NI ? 1 : 0;
    wat[i] =
        sp_place(min(r - half * NO * 16, N - 1 - n0) + half * apart, r, K);
  }
#pragma unroll
  for (int i = 0; i < XG; ++i) {
    const int r = i * 8 + (lane >> 3);
    xat[i] = sp_place(min(r, M - 1), r, K);
  }
  // Afterwards each wave goes on with a share of the tiles.
  constexpr int T = P::T;
  constexpr int TN = P::TN;
  constexpr int TO = NO * MT;
  constexpr int PER = (TO + WV - 1) / WV;
  constexpr int H = PAIR ? 2 : 1;
  s16x4 residual[PER];
  s16x4 bias[PER][2];   // (of turned pairs)
  f32x4 cos[PER], sin[PER];
  int64_t slot = 0;
  auto early = [&] {
    if constexpr (PAIR == SINGLE && !NORM) {
      if (beside.residual == nullptr) return;
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int t = min(u * WV + wave, TO - 1);
        const int row = min((t % MT) * 16 + l16, M - 1);
        const int col = min(n0 + (t / MT) * 16 + l4 * 4, N - 4);
        residual[u] = *reinterpret_cast<const s16x4*>(
            beside.residual + (int64_t)row * N + col);
      }
    }
    if constexpr (PAIR == ROPE) {
      // By way of the scalar cache: a wait for a load would be one for the
      // fills before it.
      static_assert(WV % MT == 0, "a wave's tiles are of the same rows");
      const int r0 = wave % MT * 16;
      int pos = 0;
#pragma unroll
      for (int r = 0; r < (XG == 1 ? 8 : 16); ++r) {
        const int p = load_uniform(reinterpret_cast<const int*>(
            heads.positions + min(r0 + r, M - 1)));
        if (l16 == r) pos = p;
      }
      slot = heads.slots[min(r0 + l16, M - 1)];
      const float* turn = heads.cos_sin + (int64_t)pos * (2 * heads.half);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int t = min(u * WV + wave, TO - 1);
        const int p = n0 - head * heads.half + (t / MT) * 16 + l4 * 4;
        cos[u] = *reinterpret_cast<const f32x4*>(turn + p);
        sin[u] = *reinterpret_cast<const f32x4*>(turn + heads.half + p);
        if (beside.bias != nullptr) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            bias[u][h] = *reinterpret_cast<const s16x4*>(
                beside.bias + (2 * head + h) * heads.half + p);
        }
      }
    }
  };
  const int steps = K / SP_K;
  P::run(lds, wave, steps * part / parts, steps * (part + 1) / parts,
         blockIdx.x / 8, reinterpret_cast<const char*>(w + (int64_t)w0 * K),
         wat, reinterpret_cast<const char*>(x), xat,
         reinterpret_cast<const char*>(beside.gains), early);

  f32x4 v[PER][H];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = u * WV + wave;
    if (t >= TO) break;
#pragma unroll
    for (int h = 0; h < H; ++h) v[u][h] = P::sum(lds, h * TO + t);
  }
  f32x4 squares = {0.f, 0.f, 0.f, 0.f};   // of four groups of 16 rows
  if constexpr (NORM) squares = P::sum(lds, T);
  if (parts > 1) {
    f32x4* sums = part_sums + (int64_t)tile * parts * TN * WAVE_SIZE + lane;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int t = u * WV + wave;
      if (t >= TO) break;
#pragma unroll
      for (int h = 0; h < H; ++h)
        part_put(sums + (part * TN + h * TO + t) * WAVE_SIZE, v[u][h]);
    }
    if (NORM && wave == 0)
      part_put(sums + (part * TN + T) * WAVE_SIZE, squares);
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
            p[q] = part_get(at + min(q, parts - 1) * (TN * WAVE_SIZE));
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
    if constexpr (NORM) {
      f32x4 p[SL_PARTS];
#pragma unroll
      for (int q = 0; q < SL_PARTS; ++q)
        p[q] = part_get(sums + (min(q, parts - 1) * TN + T) * WAVE_SIZE);
      squares = p[0];
#pragma unroll
      for (int q = 1; q < SL_PARTS; ++q)
        if (q < parts) squares += p[q];
    }
  }
  f32x4 roots;
#pragma unroll
  for (int j = 0; j < MT; ++j) roots[j] = rsqrtf(squares[j] / K + beside.eps);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = u * WV + wave;
    if (t >= TO) break;
    const int row = (t % MT) * 16 + l16;
    const int col = n0 + (t / MT) * 16 + l4 * 4;
    f32x4 o = v[u][0];
    if constexpr (NORM) {
      float root = roots[0];
#pragma unroll
      for (int j = 1; j < MT; ++j) root = t % MT == j ? roots[j] : root;
#pragma unroll
      for (int h = 0; h < H; ++h) v[u][h] *= root;
      o = v[u][0];
    }
    if constexpr (PAIR == SILU) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[r] = o[r] / (1.f + __expf(-o[r])) * v[u][1][r];
    }
    if (row >= M || col >= N || (XG == 1 && l16 >= 8)) continue;
    if constexpr (PAIR == ROPE) {
      const int half = heads.half, p = col - head * half;
      int2 to[2];
      float y[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4 z = v[u][h];
        if (beside.bias != nullptr) {
#pragma unroll
          for (int r = 0; r < 4; ++r) z[r] += to_f32<Tag>(bias[u][h][r]);
        }
        // Rounded as a product of its own would leave them.
        to[h] = int2{pack2<Tag>(z[0], z[1]), pack2<Tag>(z[2], z[3])};
        y[h][0] = unpack_lo<Tag>(to[h].x);
        y[h][1] = unpack_hi<Tag>(to[h].x);
        y[h][2] = unpack_lo<Tag>(to[h].y);
        y[h][3] = unpack_hi<Tag>(to[h].y);
      }
      if (head < heads.q_heads + heads.kv_heads) {
        float a[4], b[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          a[r] = __builtin_fmaf(y[0][r], cos[u][r], -(y[1][r] * sin[u][r]));
          b[r] = __builtin_fmaf(y[0][r], sin[u][r], y[1][r] * cos[u][r]);
        }
        to[0] = int2{pack2<Tag>(a[0], a[1]), pack2<Tag>(a[2], a[3])};
        to[1] = int2{pack2<Tag>(b[0], b[1]), pack2<Tag>(b[2], b[3])};
      }
      if (head < heads.q_heads) {
        short* q = out + ((int64_t)row * heads.q_heads + head) * (2 * half) + p;
        *reinterpret_cast<int2*>(q) = to[0];
        *reinterpret_cast<int2*>(q + half) = to[1];
        continue;
      }
      if (slot < 0) continue;   // padding
      const bool value = head >= heads.q_heads + heads.kv_heads;
      const int kvh = head - heads.q_heads - (value ? heads.kv_heads : 0);
      const int64_t at = (value ? heads.plane : 0) + p +
                         ((slot / heads.block_size * heads.kv_heads + kvh) *
                              heads.block_size + slot % heads.block_size) *
                             (2 * half);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (heads.fp8) {
          const uint32_t x0 = f32_to_fp8_e4m3(unpack_lo<Tag>(to[h].x));
          const uint32_t x1 = f32_to_fp8_e4m3(unpack_hi<Tag>(to[h].x));
          const uint32_t x2 = f32_to_fp8_e4m3(unpack_lo<Tag>(to[h].y));
          const uint32_t x3 = f32_to_fp8_e4m3(unpack_hi<Tag>(to[h].y));
          *reinterpret_cast<uint32_t*>((uint8_t*)heads.kv_cache + at +
                                       h * half) =
              x0 | x1 << 8 | x2 << 16 | x3 << 24;
        } else {
          *reinterpret_cast<int2*>((short*)heads.kv_cache + at + h * half) =
              to[h];
        }
      }
      continue;
    }
    if (PAIR == SINGLE && beside.bias != nullptr) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] += to_f32<Tag>(beside.bias[col + r]);
    }
    if (PAIR == SINGLE && !NORM && beside.residual != nullptr) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] += to_f32<Tag>(residual[u][r]);
    }
    *reinterpret_cast<int2*>(out + (int64_t)row * N + col) =
        int2{pack2<Tag>(o[0], o[1]), pack2<Tag>(o[2], o[3])};
  }
}

struct Plan { int form, parts; double us; };

// Form and parts of K by an estimate of the time. Its terms (added as fourth
// powers): weights at 6 TB/s; all that enters workgroups, x again in each, at
// 15 TB/s; what the fullest CU takes in at 60 GB/s, evened out by two fifths
// where neighbours still run. A workgroup's start costs 0.2 us of its CU,
// splitting K 1.5 us and the traffic of partial sums. These are coefficients
// of a fit and not bounds (the first is passed by a tenth): they come closest
// to the best of all forms over 15 layers of 2112 x 7168 to 128256 x 4096 at 1
// to 64 rows, 1.3 % from it on average, 7 % at most.
// half: 0, or columns of half a head, which tiles must not pass.
Plan plan(int xg, int64_t rows_w, int K, bool silu, bool norm = false,
          int half = 0) {
  Plan best{-1, 1, 1e30};
  auto fourth = [](double v) { return v * v * v * v; };
  for (int i = 0; i < SL_NFORMS; ++i) {
    const Form f = SL_FORMS[i];
    // Two waves have too little on the way where four fit, and are slow to
    // multiply rows by gains (4096 x 27648 with the rotation, 33 rows 47.7 us
    // in launches and 54.9 in one).
    if ((f.wv == 2 && (xg < 8 || norm)) || ((silu || half > 0) && f.ni % 2 != 0) ||
        (half > 0 && half % (f.ni * 8) != 0))
      continue;
    const int64_t tiles = (rows_w + f.ni * 16 - 1) / (f.ni * 16);
    for (int parts : {1, 2, 3, 4, 6, 8}) {
      if (parts > 1 && (tiles > SL_JOBS || tiles * parts > 1100 ||
                        K / SP_K / parts < f.wv))
        continue;
      const int lds = lds_bytes(f, xg, norm ? ceil_div(K / SP_K, parts) : 0);
      if (lds > SL_LDS) continue;
      const double mb = (f.ni * 16 + xg * 8) * 2e-6 * K / parts;
      const double jobs = (double)(tiles * parts);
      const double cus = (double)((tiles * parts + 255) / 256);
      const double load =
          cus > 1 && lds * 2 > SL_LDS
              ? cus
              : 0.6 * cus + 0.4 * std::max(1.0, jobs / 256);
      double t = std::sqrt(std::sqrt(fourth(rows_w * 2e-6 * K / 6.0) +
                                     fourth(jobs * mb / 15.0) +
                                     fourth(load * mb / 0.06))) +
                 0.2 * jobs / 256;
      if (parts > 1) t += 1.5 + 0.04 * parts * f.ni * xg;
      if (t < best.us) best = {i, parts, t};
    }
  }
  return best;
}

template <typename Tag, int I, int XG, int PAIR, bool NORM>
void launch_form(torch::Tensor& out, const torch::Tensor& x,
                 const torch::Tensor& w, const Beside& beside,
                 const Heads& heads, int N, int parts) {
  constexpr Form f = SL_FORMS[I];
  if constexpr (lds_bytes(f, XG, NORM) <= SL_LDS &&
                (f.wv > 2 || (XG == 8 && !NORM)) &&
                (!PAIR || f.ni % 2 == 0)) {
    const int lds =
        lds_bytes(f, XG, NORM ? ceil_div((int)x.size(1) / SP_K, parts) : 0);
    const int M = (int)x.size(0), K = (int)x.size(1);
    const int cols = f.ni * 16 / (PAIR ? 2 : 1);
    const int tiles = ceil_div(N, cols);
    torch::Tensor sums, arrived;
    if (parts > 1) {
      sums = torch::empty({(int64_t)tiles * parts *
                           (f.ni * ((XG + 1) / 2) + NORM) * WAVE_SIZE * 4},
                          x.options().dtype(torch::kFloat));
      arrived = arrival_counters(x, tiles);
    }
    hipLaunchKernelGGL(
        (stream_linear_kernel<Tag, f.ni, XG, f.wv, f.d, PAIR, NORM>),
        dim3(tiles * parts), dim3(f.wv * WAVE_SIZE), lds,
        c10::hip::getCurrentHIPStream().stream(), (short*)out.data_ptr(),
        (const short*)x.data_ptr(), (const short*)w.data_ptr(), beside, heads,
        M, N, K, tiles, parts, parts > 1 ? (f32x4*)sums.data_ptr() : nullptr,
        parts > 1 ? (unsigned*)arrived.data_ptr() : nullptr);
  } else {
    TORCH_CHECK(false, "stream_linear: form does not fit");
  }
}

template <typename Tag, int PAIR, bool NORM = false>
void launch(torch::Tensor& out, const torch::Tensor& x,
            const torch::Tensor& w, const Beside& beside, int N,
            const Heads& heads = Heads{}) {
  const int xg = row_groups(x.size(0));
  const Plan p = plan(xg, w.size(0), (int)x.size(1), PAIR == SILU, NORM,
                      heads.half);
  auto by_rows = [&](auto form) {
    constexpr int I = decltype(form)::value;
    auto groups = [&](auto n) {
      launch_form<Tag, I, decltype(n)::value, PAIR, NORM>(
          out, x, w, beside, heads, N, p.parts);
    };
    if (xg == 1) groups(std::integral_constant<int, 1>{});
    else if (xg == 2) groups(std::integral_constant<int, 2>{});
    else if (xg == 4) groups(std::integral_constant<int, 4>{});
    else groups(std::integral_constant<int, 8>{});
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

// x, w and what is beside them as stream_linear_takes and the callers have
// checked them.
static torch::Tensor stream_linear_beside(const torch::Tensor& x,
                                          const torch::Tensor& w,
                                          const Beside& beside) {
  const int64_t N = w.size(0);
  auto out = torch::empty({x.size(0), N}, x.options());
  if (x.scalar_type() == torch::kBFloat16)
    launch<BF16Tag, SINGLE>(out, x, w, beside, (int)N);
  else
    launch<FP16Tag, SINGLE>(out, x, w, beside, (int)N);
  HIP_CHECK_KERNEL();
  return out;
}

torch::Tensor stream_linear(const torch::Tensor& x, const torch::Tensor& w,
                            const c10::optional<torch::Tensor>& bias) {
  Beside beside;
  if (bias.has_value()) beside.bias = (const short*)bias->data_ptr();
  return stream_linear_beside(x, w, beside);
}

// (An operand elsewhere would be read by its address there.)
static void check_device(const torch::Tensor& a,
                         std::initializer_list<const torch::Tensor*> others,
                         const c10::optional<torch::Tensor>& bias) {
  for (const torch::Tensor* t : others)
    TORCH_CHECK(t->device() == a.device(), "operands on ", t->device(),
                " and ", a.device());
  TORCH_CHECK(!bias.has_value() || bias->device() == a.device(),
              "operands on ", bias->device(), " and ", a.device());
}

// A product by itself. (Rows that are not multiples of 16 B fall outside the
// aligned kernels, the library's own among them.)
static torch::Tensor product(const torch::Tensor& x, const torch::Tensor& w,
                             const c10::optional<torch::Tensor>& bias) {
  const int64_t per16 = 16 / x.element_size();
  if (w.size(0) % per16 != 0 || w.size(1) % per16 != 0)
    return at::linear(x, w, bias);
  return lt_linear(x, w, bias);
}

static bool bias_fits(const c10::optional<torch::Tensor>& bias,
                      const torch::Tensor& w) {
  return !bias.has_value() ||
         (bias->scalar_type() == w.scalar_type() && bias->is_contiguous() &&
          bias->numel() == w.size(0));
}

// a @ w^T + bias + residual; in one launch, rounded once, where this file
// takes the product.
torch::Tensor linear_add(torch::Tensor a, torch::Tensor w,
                         c10::optional<torch::Tensor> bias,
                         torch::Tensor residual) {
  TORCH_CHECK(a.dim() == 2 && w.dim() == 2 && a.size(1) == w.size(1) &&
                  a.scalar_type() == w.scalar_type() &&
                  residual.dim() == 2 && residual.size(0) == a.size(0) &&
                  residual.size(1) == w.size(0) &&
                  residual.scalar_type() == a.scalar_type(),
              "linear_add: [M, K] x [N, K] + [M, N]");
  check_device(a, {&w, &residual}, bias);
  auto x = a.contiguous();
  if (x.size(0) == 0 || !residual.is_contiguous() ||
      (uintptr_t)residual.data_ptr() % 8 != 0 || !bias_fits(bias, w))
    return product(x, w, bias) + residual;
  const bool tiles = !bias.has_value() &&
                     tile_linear_first(x.size(0), w.size(0), x.size(1), false);
  if (tiles || !stream_linear_takes(x, w, w.size(0))) {
    auto out = torch::empty({x.size(0), w.size(0)}, x.options());
    if (!bias.has_value() &&
        tile_linear_add(out, x, w, false, (const short*)residual.data_ptr()))
      return out;
    return product(x, w, bias) + residual;
  }
  Beside beside;
  if (bias.has_value()) beside.bias = (const short*)bias->data_ptr();
  beside.residual = (const short*)residual.data_ptr();
  return stream_linear_beside(x, w, beside);
}

// Whether the norm of `rows` rows goes with the product (bf16 only: fp16 rows
// times gains may pass 65504 where normalized ones do not). Up to 32 rows, if
// the gains leave room for the form that the product takes without them. us with
// the launches that go, and in one (4096 x 6144 with the rotation, 4096 x 28672
// and 3584 x 37888 with the activation): 8 rows 16.0 and 12.0, 38.0 and 35.5,
// 48.0 and 45.9; 32 rows 19.1 and 14.4, 39.5 and 41.4 (another form: not
// taken), 53.1 and 51.5; 64 rows 22.8 and 18.8, tiles, and two waves.
//
// half: columns of half a head, if the rotation goes with the product too. Then
// up to 64 rows in that form. Heads whose halves its tiles do not fit (64
// columns, and 96 weight rows of a tile) take another one. That may cost more
// than the launches, up to 60 % of the product, and where depends on how tiles
// come out on 256 CUs, which the estimate knows to 2 us at best. So other forms
// are taken, unless the estimate is that far behind, by what held for 139 of
// 141 products of 128 to 12288 columns (two lost 3 %). us apart and in one:
//  * K split over workgroups: 10240 x 8192, 33 and 64 rows 43.3 and 43.3, 46.6
//    and 44.7; 3840 x 11840, 16 rows 26.6 and 20.5. (Not split, of narrow
//    layers: 4096 x 7680, 1 row 17.6 and 20.1.)
//  * wider tiles: 24576 x 8192, 16 rows 76.1 and 61.8. (Narrower ones: 18432 x
//    4096, 8 rows 30.7 and 34.5.)
//  * 32 weight rows for 64, up to 32 rows: 9216 x 3072 (heads of 96), 16 and 32
//    rows 19.6 and 17.2, 21.7 and 20.6. (64 rows 25.9 and 36.4.)
//  * up to 16 rows of up to 2048 columns, where launches are most of the time:
//    2304 x 768 8.9 and 5.1.
static bool norm_sizes(int64_t rows, int64_t weight_rows, int64_t k,
                       bool silu, int half = 0) {
  if (tile_linear_first(rows, weight_rows, k, silu) ||
      !stream_sizes(rows, weight_rows, silu ? weight_rows / 2 : weight_rows,
                    k))
    return false;
  const int xg = row_groups(rows);
  const Plan with = plan(xg, weight_rows, (int)k, silu, true, half);
  const Plan without = plan(xg, weight_rows, (int)k, silu);
  if (with.form < 0) return false;
  if (with.form == without.form && with.parts == without.parts)
    return half > 0 || rows <= 32;
  const Form f = SL_FORMS[with.form], other = SL_FORMS[without.form];
  return half > 0 && with.us < without.us + 2 &&
         (with.parts > 1 || (f.ni > other.ni && other.ni > 1) ||
          (f.ni == 2 && other.ni == 4 && rows <= 32) ||
          (k <= 2048 && rows <= 16));
}

// What a product of these sizes runs as, for 16-bit operands that begin on
// 16 B: {0} the library, {1, 16-row groups of weights, waves, ring steps,
// 8-row groups of x, parts of K} stream_linear, {2, weight rows of a tile,
// parts of K} tile_linear. norm: of a norm's rows, with half a head's columns
// where heads turn as a whole; {0} where the norm is a launch of its own.
std::vector<int64_t> linear_form(int64_t rows, int64_t weight_rows, int64_t k,
                                 bool silu, bool norm, int64_t half) {
  const int64_t n = silu ? weight_rows / 2 : weight_rows;
  if (norm && !norm_sizes(rows, weight_rows, k, silu, (int)half)) return {0};
  if (!tile_linear_first(rows, weight_rows, k, silu) &&
      stream_sizes(rows, weight_rows, n, k)) {
    const int xg = row_groups(rows);
    const Plan p = plan(xg, weight_rows, (int)k, silu, norm, (int)half);
    const Form f = SL_FORMS[p.form];
    return {1, f.ni, f.wv, f.d, xg, p.parts};
  }
  const TileForm tile = tile_linear_form(rows, weight_rows, k, silu);
  if (tile.cols == 0) return {0};
  return {2, tile.cols, tile.parts};
}

// Whether the residual goes with the product, without a bias.
static bool add_sizes(int64_t rows, int64_t weight_rows, int64_t k) {
  if (tile_linear_first(rows, weight_rows, k, false))
    return tile_linear_form(rows, weight_rows, k, false).parts > 1;
  return stream_sizes(rows, weight_rows, weight_rows, k);
}

// Whether a decoder layer of up to 64 rows has fewer launches if products take
// its norms, sums and rotation along: `qkv` and `gate_up` weight rows on norms
// of `hidden` columns, products back to them from `heads` and `inner` columns,
// heads of twice `half` columns that turn as a whole (0: others). Sums must be
// epilogues, or launches would only move; a norm may stay one.
bool layer_streams(int64_t rows, int64_t hidden, int64_t qkv, int64_t heads,
                   int64_t gate_up, int64_t inner, int64_t half) {
  return gate_up == 2 * inner && rows > 0 && rows <= SL_ROWS &&
         add_sizes(rows, hidden, heads) && add_sizes(rows, hidden, inner) &&
         (norm_sizes(rows, qkv, hidden, false, (int)half) ||
          norm_sizes(rows, gate_up, hidden, true));
}

// linear (or, silu, linear_silu_and_mul) of rms_norm(a, gains, eps); in one
// launch where norm_sizes says so.
torch::Tensor norm_linear(torch::Tensor a, torch::Tensor gains, double eps,
                          torch::Tensor w, c10::optional<torch::Tensor> bias,
                          bool silu) {
  TORCH_CHECK(a.dim() == 2 && w.dim() == 2 && a.size(1) == w.size(1) &&
                  a.scalar_type() == w.scalar_type() && gains.dim() == 1 &&
                  gains.size(0) == a.size(1) &&
                  gains.scalar_type() == a.scalar_type(),
              "norm_linear: [M, K] x [N, K], gains [K]");
  check_device(a, {&gains, &w}, bias);
  TORCH_CHECK(!silu || (w.size(0) % 2 == 0 && !bias.has_value()),
              "norm_linear: the activation takes [gate; up] without a bias");
  auto x = a.contiguous();
  const int64_t N = silu ? w.size(0) / 2 : w.size(0);
  if (x.scalar_type() != torch::kBFloat16 || x.size(0) == 0 ||
      !gains.is_contiguous() || (uintptr_t)gains.data_ptr() % 16 != 0 ||
      !bias_fits(bias, w) || !stream_linear_takes(x, w, N) ||
      !norm_sizes(x.size(0), w.size(0), x.size(1), silu)) {
    auto y = rms_norm(x, gains, eps);
    if (!silu) return product(y, w, bias);
    if (w.size(0) % 16 == 0 && w.size(1) % 8 == 0)
      return linear_silu_and_mul(y, w);
    return silu_and_mul_any(product(y, w, c10::nullopt));
  }
  Beside beside;
  if (bias.has_value()) beside.bias = (const short*)bias->data_ptr();
  beside.gains = (const short*)gains.data_ptr();
  beside.eps = (float)eps;
  auto out = torch::empty({x.size(0), N}, x.options());
  if (silu) launch<BF16Tag, SILU, true>(out, x, w, beside, (int)N);
  else      launch<BF16Tag, SINGLE, true>(out, x, w, beside, (int)N);
  HIP_CHECK_KERNEL();
  return out;
}

// Queries of rms_norm(a, gains, eps) @ w^T (+ bias), w = [q heads; k heads; v
// heads], rotated over all of a head, with the rotated keys and the values in
// the cache; in one launch where norm_sizes says so of tiles within a head's
// halves, else as the steps it stands for. [M, q_heads, D], whose rows may lie
// apart.
torch::Tensor norm_qkv_rope_cache(
    torch::Tensor a, torch::Tensor gains, double eps, torch::Tensor w,
    c10::optional<torch::Tensor> bias, torch::Tensor positions,
    torch::Tensor slots, torch::Tensor cos_sin, torch::Tensor kv_cache) {
  TORCH_CHECK(a.dim() == 2 && w.dim() == 2 && a.size(1) == w.size(1) &&
                  kv_cache.dim() == 5 && kv_cache.size(0) == 2 &&
                  kv_cache.is_contiguous(),
              "norm_qkv_rope_cache: [M, K] x [rows, K], cache [2, blocks, "
              "heads, block, D]");
  const int64_t M = a.size(0), D = kv_cache.size(4), Hkv = kv_cache.size(2);
  const int64_t Hq = w.size(0) / D - 2 * Hkv;
  TORCH_CHECK(Hq > 0 && w.size(0) == (Hq + 2 * Hkv) * D,
              "norm_qkv_rope_cache: rows of w are heads");
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 &&
                  cos_sin.is_contiguous() && cos_sin.dim() == 2 &&
                  cos_sin.size(1) == D &&
                  positions.scalar_type() == torch::kInt64 &&
                  slots.scalar_type() == torch::kInt64 &&
                  positions.is_contiguous() && slots.is_contiguous() &&
                  positions.numel() >= M && slots.numel() >= M,
              "norm_qkv_rope_cache: fp32 table [positions, D], int64 "
              "positions and slots");
  TORCH_CHECK(kv_cache.scalar_type() == a.scalar_type() ||
                  kv_cache.scalar_type() == torch::kFloat8_e4m3fn,
              "norm_qkv_rope_cache: cache of the rows' type or e4m3");
  check_device(a, {&gains, &w, &positions, &slots, &cos_sin, &kv_cache}, bias);
  auto x = a.contiguous();
  const int half = (int)D / 2;
  if (x.scalar_type() != torch::kBFloat16 ||
      gains.scalar_type() != torch::kBFloat16 || gains.numel() != x.size(1) ||
      !gains.is_contiguous() || (uintptr_t)gains.data_ptr() % 16 != 0 ||
      (uintptr_t)cos_sin.data_ptr() % 16 != 0 ||
      (uintptr_t)kv_cache.data_ptr() % 16 != 0 || D % 32 != 0 ||
      !bias_fits(bias, w) ||
      (bias.has_value() && (uintptr_t)bias->data_ptr() % 8 != 0) || M == 0 ||
      !stream_linear_takes(x, w, w.size(0)) ||
      !norm_sizes(M, w.size(0), x.size(1), false, half)) {
    auto qkv = norm_linear(x, gains, eps, w, bias, false);
    auto rows = qkv.view({M, Hq + 2 * Hkv, D});
    auto q = rows.narrow(1, 0, Hq);
    rope_and_cache(positions, q, rows.narrow(1, Hq, Hkv),
                   rows.narrow(1, Hq + Hkv, Hkv), cos_sin, D, kv_cache, slots);
    return q;
  }
  Beside beside;
  if (bias.has_value()) beside.bias = (const short*)bias->data_ptr();
  beside.gains = (const short*)gains.data_ptr();
  beside.eps = (float)eps;
  Heads heads;
  heads.positions = positions.data_ptr<int64_t>();
  heads.slots = slots.data_ptr<int64_t>();
  heads.cos_sin = cos_sin.data_ptr<float>();
  heads.kv_cache = kv_cache.data_ptr();
  heads.plane = kv_cache.stride(0);
  heads.half = half;
  heads.q_heads = (int)Hq;
  heads.kv_heads = (int)Hkv;
  heads.block_size = (int)kv_cache.size(3);
  heads.fp8 = kv_cache.scalar_type() == torch::kFloat8_e4m3fn;
  auto out = torch::empty({M, Hq, D}, x.options());
  launch<BF16Tag, ROPE, true>(out, x, w, beside, (int)(w.size(0) / 2), heads);
  HIP_CHECK_KERNEL();
  return out;
}

// silu(x @ gate^T) * (x @ up^T), w = [gate; up]; in one launch where this file
// or tile_linear takes it (the products are then not rounded in between).
torch::Tensor linear_silu_and_mul(torch::Tensor a, torch::Tensor w) {
  TORCH_CHECK(w.dim() == 2 && w.size(0) % 2 == 0 && a.dim() >= 1 &&
              a.size(-1) == w.size(1) && a.scalar_type() == w.scalar_type(),
              "linear_silu_and_mul: [.., K] x [2N, K]");
  check_device(a, {&w}, c10::nullopt);
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
    launch<BF16Tag, SILU>(out, x, w, Beside{}, (int)N);
  else
    launch<FP16Tag, SILU>(out, x, w, Beside{}, (int)N);
  HIP_CHECK_KERNEL();
  return out.reshape(sizes);
}

}  // namespace vllm_amd
