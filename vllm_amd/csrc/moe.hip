// MoE grouped-GEMM kernels for CDNA4 (gfx950).
//
// Role of the reference's Triton grouped GEMM
// (vllm/model_executor/layers/fused_moe/fused_moe.py:299) and
// moe_align_block_size (csrc/libtorch_stable/moe/moe_align_sum_kernels.cu:326),
// as hand-written MFMA kernels: (token, slot) rows are sorted by expert
// into tiles on the device (no host sync; shapes depend only on (T, topk,
// E), so the whole layer is hipGraph-capturable), then two products run
// over the tiles. The activation is the first product's epilogue: gate
// and up rows of the same columns belong to one workgroup.
//
// Two forms of the product, chosen by the average number of rows an
// expert gets (ops/hip_ops.py):
//   moe_rows_kernel    few rows: every weight is read once and used for at
//                      most 64 rows, so HBM bounds it.
//   moe_stream_kernel  the same for weights stored in fragment order
//                      ([E][N/16][K/32][64 lanes][8], ops/hip_ops.py
//                      moe_shuffle_weights), or that do not begin on 16 B:
//                      straight into MFMA fragments, no LDS in the loop.
//   moe_tiles.hip      many rows: the matrix cores bound it; 128 or 256 x
//                      256 tiles through LDS.
//
// Pipeline (ops/hip_ops.py fused_moe):
//   moe_align: counts -> tile-aligned offsets -> sorted flat ids + the
//              inverse permutation (combine is deterministic)
//   moe_gemm(hidden, w13) + activation -> act [EM, I] (rows gathered)
//   moe_gemm(act, w2)                  -> y [EM, H]   (rows in tile order)
//   moe_combine: out[t] = sum_k w[t,k] * y[inv_perm[t*K+k]]

#include <torch/all.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include "moe_rows.h"
#include "tile_product.h"

namespace vllm_amd {

namespace moe {

constexpr int BM = 64;    // token rows per tile of the few-row kernels
constexpr int THREADS = 256;
constexpr int SENTINEL = 0x7fffffff;
constexpr int LDS_EXPERTS = 1024;   // whose counters fit LDS

// --------------------------------------------------------------------------
// Alignment. Counting and placing with one atomic per row on global
// counters costs 113 us at 32768 rows (every row of an expert waits for
// the one before); counters in LDS, one set per block of 2048 rows, and a
// prefix over the blocks cost 13 us (32 while a thread by itself filled up
// its expert's last tile and read the blocks' counts one by one). Up to 2048
// rows one workgroup does it all in one launch (48 rows on 8 experts: 6.5 ->
// 3.6 us). Counters of more than 1024 experts (LDS false) are in the scratch
// instead, one set per block all the same.
constexpr int ALIGN_ROWS = 2048;   // rows per block

// counts[e] -> off[e] = first row of expert e in tile order, and what the
// products read per tile. Called by all THREADS threads of one workgroup.
DEVINL void place_experts(const int* counts, int* off, int e, int bm,
                          int* __restrict__ expert_tiles, int max_tiles,
                          int* __restrict__ sorted, int* scan) {
  const int tid = threadIdx.x;
  const int per = (e + THREADS - 1) / THREADS;
  int tiles = 0;
  for (int i = tid * per; i < min(e, (tid + 1) * per); ++i)
    tiles += (counts[i] + bm - 1) / bm;
  scan[tid] = tiles;
  __syncthreads();
  for (int d = 1; d < THREADS; d <<= 1) {
    const int v = tid >= d ? scan[tid - d] : 0;
    __syncthreads();
    scan[tid] += v;
    __syncthreads();
  }
  int t = scan[tid] - tiles;
  const int total = scan[THREADS - 1];
  for (int i = tid * per; i < min(e, (tid + 1) * per); ++i) {
    const int n = counts[i];
    off[i] = t * bm;
    for (int k = 0; k < n; k += bm) expert_tiles[t++] = i;
  }
  for (int i = total + tid; i < max_tiles; i += THREADS) expert_tiles[i] = -1;
  if (tid == 0) expert_tiles[max_tiles] = total;
  __syncthreads();
  // What the last tiles of experts hold no row in: 16 lanes an expert.
  for (int i = tid / 16; i < e; i += THREADS / 16) {
    const int n = counts[i], end = (n + bm - 1) / bm * bm;
    for (int k = n + tid % 16; k < end; k += 16)
      sorted[off[i] + k] = SENTINEL;
  }
  __syncthreads();
}

template <bool LDS>
__global__ __launch_bounds__(THREADS) void align_small_kernel(
    const int* __restrict__ ids, int total, int e, int bm,
    int* __restrict__ expert_tiles, int max_tiles, int* __restrict__ sorted,
    int* __restrict__ inv_perm, int* counters) {
  __shared__ int lds[LDS ? 2 * LDS_EXPERTS : 1], scan[THREADS];
  int* counts = LDS ? lds : counters;
  int* off = counts + (LDS ? LDS_EXPERTS : e);
  for (int i = threadIdx.x; i < e; i += THREADS) counts[i] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < total; i += THREADS)
    atomicAdd(&counts[ids[i]], 1);
  __syncthreads();
  place_experts(counts, off, e, bm, expert_tiles, max_tiles, sorted, scan);
  for (int i = threadIdx.x; i < total; i += THREADS) {
    const int pos = atomicAdd(&off[ids[i]], 1);
    sorted[pos] = i;
    inv_perm[i] = pos;
  }
}

// part[b][e]: rows of expert e in block b.
template <bool LDS>
__global__ __launch_bounds__(THREADS) void align_count_kernel(
    const int* __restrict__ ids, int total, int e, int* part) {
  __shared__ int lds[LDS ? LDS_EXPERTS : 1];
  int* counts = LDS ? lds : part + (int64_t)blockIdx.x * e;
  for (int i = threadIdx.x; i < e; i += THREADS) counts[i] = 0;
  __syncthreads();
  const int end = min(total, ((int)blockIdx.x + 1) * ALIGN_ROWS);
  for (int i = blockIdx.x * ALIGN_ROWS + threadIdx.x; i < end; i += THREADS)
    atomicAdd(&counts[ids[i]], 1);
  if constexpr (LDS) {
    __syncthreads();
    for (int i = threadIdx.x; i < e; i += THREADS)
      part[(int64_t)blockIdx.x * e + i] = counts[i];
  }
}

// part[b][e] -> first row of block b's rows of expert e.
template <bool LDS>
__global__ __launch_bounds__(THREADS) void align_place_kernel(
    int* __restrict__ part, int blocks, int e, int bm,
    int* __restrict__ expert_tiles, int max_tiles, int* __restrict__ sorted,
    int* counters) {
  __shared__ int lds[LDS ? 2 * LDS_EXPERTS : 1], scan[THREADS];
  int* counts = LDS ? lds : counters;
  int* off = counts + (LDS ? LDS_EXPERTS : e);
  for (int i = threadIdx.x; i < e; i += THREADS) {
    int n = 0;
#pragma unroll 8
    for (int b = 0; b < blocks; ++b) n += part[(int64_t)b * e + i];
    counts[i] = n;
  }
  __syncthreads();
  place_experts(counts, off, e, bm, expert_tiles, max_tiles, sorted, scan);
  for (int i = threadIdx.x; i < e; i += THREADS) {
    int at = off[i];
    for (int b0 = 0; b0 < blocks; b0 += 8) {   // loads of eight at a time
      int n[8];
#pragma unroll
      for (int b = 0; b < 8; ++b)
        n[b] = b0 + b < blocks ? part[(int64_t)(b0 + b) * e + i] : 0;
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        if (b0 + b < blocks) part[(int64_t)(b0 + b) * e + i] = at;
        at += n[b];
      }
    }
  }
}

template <bool LDS>
__global__ __launch_bounds__(THREADS) void align_scatter_kernel(
    const int* __restrict__ ids, int total, int e, int* part,
    int* __restrict__ sorted, int* __restrict__ inv_perm) {
  __shared__ int lds[LDS ? LDS_EXPERTS : 1];
  int* off = LDS ? lds : part + (int64_t)blockIdx.x * e;
  if constexpr (LDS) {
    for (int i = threadIdx.x; i < e; i += THREADS)
      off[i] = part[(int64_t)blockIdx.x * e + i];
    __syncthreads();
  }
  const int end = min(total, ((int)blockIdx.x + 1) * ALIGN_ROWS);
  for (int i = blockIdx.x * ALIGN_ROWS + threadIdx.x; i < end; i += THREADS) {
    const int pos = atomicAdd(&off[ids[i]], 1);
    sorted[pos] = i;
    inv_perm[i] = pos;
  }
}

// --------------------------------------------------------------------------
// Into how many parts the column blocks go: three or more blocks each and
// no more than a tenth of unevenness, more only where row tiles are few.
// Measured in 8 / 4 / 2 / 1 parts, ms: 8 experts, 4096 x 14336 (112 and 16
// blocks), 96 rows 0.63 / 0.67 / 0.71 / 0.78; 64 experts, 7168 x 2048 (16
// and 28), 512 rows 3.33 / 3.16 / 3.16 / 3.18; 128 experts, 2048 x 768 (6
// and 8), 64 rows 0.32 / 0.32 / 0.30 / 0.30.
static int split_of_grid(int m_tiles, int n_blocks) {
  int split = 8;
  while (split > 1 && (n_blocks < 3 * split ||
                       ceil_div(n_blocks, split) * split * 10 > n_blocks * 11))
    split /= 2;
  while (split < 8 && m_tiles < 2 * (8 / split)) split *= 2;
  return split;
}

// --------------------------------------------------------------------------
// Few rows: weights are read once and used for at most 64 rows, so HBM bounds
// it; at 64 rows the matrix cores are 15 % busy, so rows of padding cost
// nothing. 8-row groups past the tile's last row are left out.
//
// Weights as they are stored: stream_product.h, 128 weight rows (64 gate + 64
// up rows for gated experts) a workgroup, or 32 where those are too few to
// fill the chip; LDS is filled in whole lines that leave L2 first. us by
// fragments, as below, and so: 8 experts of 4096 x 14336, 2 a token, 1 token
// 166 / 115, 4 409 / 330, 48 517 / 435 (6.5 TB/s), 90 592 / 444; 64 of 7168 x
// 2048, 8 a token, 64 tokens 950 / 805; 128 of 2048 x 768 195 / 179.
// Workgroups that are enough (of the tiles that there may be; few of them
// are empty). us with 128 and with 32 weight rows a workgroup: 16 experts of
// 1024 x 3584 without a gate, second product in 128 and 512, 8 tokens of two
// 47.3 and 42.1, in 136 and 544, 64 tokens 63.4 and 54.5; 8 of 1024 x 2048, first
// product in 256 and 1024, 4 tokens 24.6 and 28.9.
constexpr int SR_FILL = 192;

template <typename Tag, int ACT, int NI>
__launch_bounds__(THREADS, 1) __global__
void moe_rows_kernel(const short* __restrict__ A,
                     const short* __restrict__ W, int64_t expert_stride,
                     short* __restrict__ C, int64_t ldc,
                     const int* __restrict__ sorted,
                     const int* __restrict__ expert_tiles, int K, int N,
                     int topk_div, int total_flat, int m_tiles,
                     int n_blocks) {
  int tile, blk;
  if (!tile_of_block(m_tiles, n_blocks, tile, blk)) return;
  const int expert = expert_tiles[tile];
  if (expert < 0) return;  // padding tile
  __shared__ __align__(16) char lds[ROWS_LDS];
  const int rows = rows_of_tile<BM>(sorted, tile, total_flat);
  const int n0 = blk * (ACT == SILU_GATED ? NI * 8 : NI * 16);
  const short* w = W + expert * expert_stride;
  rows_body<Tag, ACT, NI>(lds, A, w, C, ldc, sorted, K, N, topk_div,
                          tile * BM, rows, n0);
}

// Weights in fragment order, or that do not begin on 16 B: a workgroup takes
// 64 weight rows (32 gate + 32 up rows for gated experts) of an expert and
// up to 64 token rows; its four waves take a quarter of K each and add up at
// the end. A wave reads 64 weight rows 128 B at a time straight into A
// fragments, the next 128 B while it multiplies; token rows are B fragments,
// from L2. Two workgroups per CU keep 128 KB of weights in flight.
constexpr int ST_W = 64;     // weight rows per workgroup
constexpr int ST_U = 2;      // 32-wide K steps per load

// Runs of 1 KB (fragment order) leave L2 first; of half lines the other half
// would be fetched again (519 -> 588 us for 48 tokens as above).
template <int STEP> DEVINL s16x8 weights(const short* p) {
  const s16x8* v = reinterpret_cast<const s16x8*>(p);
  return STEP > 32 ? __builtin_nontemporal_load(v) : *v;
}

template <typename Tag, int ACT, int STEP, int MT>
DEVINL void stream_body(const short* const (&wp)[4],
                        const short* const (&xp)[4], int s0, int s1,
                        f32x4* red, int wave, int lane, int rows,
                        short* __restrict__ C, int64_t ldc, int n0, int N) {
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  f32x4 acc[4][MT];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  s16x8 wf[ST_U][4], xf[ST_U][MT], wn[ST_U][4], xn[ST_U][MT];
  auto load = [&](int s, auto& w, auto& x) {
#pragma unroll
    for (int u = 0; u < ST_U; ++u) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[u][i] = weights<STEP>(wp[i] + (int64_t)(s + u) * STEP);
#pragma unroll
      for (int j = 0; j < MT; ++j)
        x[u][j] = *reinterpret_cast<const s16x8*>(xp[j] + (s + u) * 32);
    }
  };
  auto multiply = [&](auto& w, auto& x) {
#pragma unroll
    for (int u = 0; u < ST_U; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[i][j] = mfma16<Tag>(w[u][i], x[u][j], acc[i][j]);
  };
  int s = s0;
  if (s + ST_U <= s1) {
    load(s, wf, xf);
    for (; s + 2 * ST_U <= s1; s += ST_U) {
      load(s + ST_U, wn, xn);
      multiply(wf, xf);
#pragma unroll
      for (int u = 0; u < ST_U; ++u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) wf[u][i] = wn[u][i];
#pragma unroll
        for (int j = 0; j < MT; ++j) xf[u][j] = xn[u][j];
      }
    }
    multiply(wf, xf);
    s += ST_U;
  }
  for (; s < s1; ++s) {   // an odd step is left
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const s16x8 w = weights<STEP>(wp[i] + (int64_t)s * STEP);
#pragma unroll
      for (int j = 0; j < MT; ++j)
        acc[i][j] = mfma16<Tag>(
            w, *reinterpret_cast<const s16x8*>(xp[j] + s * 32), acc[i][j]);
    }
  }

#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
      red[((wave * 4 + i) * MT + j) * WAVE_SIZE + lane] = acc[i][j];
  __syncthreads();
  auto sum = [&](int i, int j) {
    f32x4 v = red[(i * MT + j) * WAVE_SIZE + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w)
      v += red[((w * 4 + i) * MT + j) * WAVE_SIZE + lane];
    return v;
  };
  // Each wave finishes a share of the 16 x 16 tiles: column l16 is a token
  // row, the four values are neighbouring columns of the output.
  constexpr int PARTS = ACT == SILU_GATED ? 2 : 4;
#pragma unroll
  for (int u = 0; u < PARTS * MT / 4 + (PARTS * MT % 4 != 0); ++u) {
    const int unit = u * 4 + wave;
    if (unit >= PARTS * MT) break;
    const int p = unit % PARTS;
    const int j = unit / PARTS;
    f32x4 v = sum(p, j);
    if constexpr (ACT == SILU_GATED) {
      const f32x4 up = sum(p + 2, j);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = silu_mul(v[r], up[r]);
    } else if constexpr (ACT == RELU2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = relu2(v[r]);
    }
    const int row = j * 16 + l16;
    const int col = n0 + p * 16 + l4 * 4;
    if (row < rows && col < N) {
      int2 o;
      o.x = pack2<Tag>(v[0], v[1]);
      o.y = pack2<Tag>(v[2], v[3]);
      *reinterpret_cast<int2*>(C + (int64_t)row * ldc + col) = o;
    }
  }
}

template <typename Tag, int ACT, bool SHUF>
__launch_bounds__(THREADS, 2) __global__
void moe_stream_kernel(const short* __restrict__ A, int64_t lda,
                       const short* __restrict__ W, int64_t expert_stride,
                       short* __restrict__ C, int64_t ldc,
                       const int* __restrict__ sorted,
                       const int* __restrict__ expert_tiles, int K, int N,
                       int topk_div, int total_flat, int m_tiles,
                       int n_blocks) {
  int tile, blk;
  if (!tile_of_block(m_tiles, n_blocks, tile, blk)) return;
  const int expert = expert_tiles[tile];
  if (expert < 0) return;  // padding tile
  __shared__ __align__(16) f32x4 red[4 * 4 * 4 * WAVE_SIZE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  const int rows = rows_of_tile<BM>(sorted, tile, total_flat);
  const int n0 = blk * (ACT == SILU_GATED ? ST_W / 2 : ST_W);

  const short* wp[4];
  const short* we = W + expert * expert_stride;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // 16 rows, whole ones: N is a multiple of 16 where SHUF.
    const int r0 = n0 + (ACT == SILU_GATED ? i & 1 : i) * 16;
    const int up = ACT == SILU_GATED ? (i >> 1) * N : 0;
    if constexpr (SHUF)
      wp[i] = we + (int64_t)(min(r0, N - 16) + up) * K + lane * 8;
    else
      wp[i] = we + (int64_t)(min(r0 + l16, N - 1) + up) * K + l4 * 8;
  }
  const short* xp[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = tile * BM + min(j * 16 + l16, rows - 1);
    xp[j] = A + (topk_div > 0 ? sorted[r] / topk_div : r) * lda + l4 * 8;
  }
  constexpr int STEP = SHUF ? 16 * 32 : 32;   // elements to the next step
  const int steps = K / 32;
  const int s0 = steps * wave / 4, s1 = steps * (wave + 1) / 4;
  short* c = C + (int64_t)tile * BM * ldc;
  if (rows <= 16)
    stream_body<Tag, ACT, STEP, 1>(wp, xp, s0, s1, red, wave, lane, rows, c,
                                   ldc, n0, N);
  else if (rows <= 32)
    stream_body<Tag, ACT, STEP, 2>(wp, xp, s0, s1, red, wave, lane, rows, c,
                                   ldc, n0, N);
  else
    stream_body<Tag, ACT, STEP, 4>(wp, xp, s0, s1, red, wave, lane, rows, c,
                                   ldc, n0, N);
}

// --------------------------------------------------------------------------
// Weighted combine: out[t, :] = sum_k w[t*K+k] * Y[inv_perm[t*K+k], :].
// Bound by memory: a workgroup is 128 chunks of 8 columns of a token, so that
// a few tokens are many workgroups, no wave is half empty and the parts of a
// row are read together; four rows are under way at a time. ONCE: what is
// read leaves the caches first; not where it is still cached from its own
// making (4096 tokens x 2 x 4096, 67 MB, 16.1 us and 18.8 so; x 8 x 7168 104.6
// and 92.8). us before (a token a workgroup, row after row) and now, K = 8:
// 64 x 7168 8.4 -> 3.3, 512 x 7168 15.1 -> 11.1, 4096 x 7168 111 -> 93, 4096 x
// 2048 29.0 -> 29.1.
constexpr int COMBINE = 128;
constexpr int64_t READ_ONCE_BYTES = 96ll << 20;

template <typename Tag, bool ONCE>
__global__ __launch_bounds__(COMBINE) void combine_kernel(
    short* __restrict__ out, const short* __restrict__ Y, long ldy,
    const float* __restrict__ weights, const int* __restrict__ inv_perm,
    int topk, int H, int parts) {
  const int t = blockIdx.x / parts;
  const int h = (blockIdx.x % parts * COMBINE + threadIdx.x) * 8;
  if (h >= H) return;
  float acc[8] = {0.f};
  const float* w = weights + (int64_t)t * topk;
  const int* at = inv_perm + (int64_t)t * topk;
#pragma unroll 4
  for (int k = 0; k < topk; ++k) {
    const s16x8 v = load16<ONCE>(Y + (long)at[k] * ldy + h);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += w[k] * to_f32<Tag>(v[j]);
  }
  s16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = from_f32<Tag>(acc[j]);
  *reinterpret_cast<s16x8*>(out + (long)t * H + h) = o;
}

}  // namespace moe

// Host-side entry points -----------------------------------------------------

// Rows per tile of the forms of the product: 0 streams weights, 1 and 2
// are the 128- and 256-row tiles.
int64_t moe_tile_rows(int64_t form) {
  TORCH_CHECK(form >= 0 && form <= 2);
  return form == 2 ? 256 : form == 1 ? 128 : moe::BM;
}

// For the tests: {XCD, row tile, column block} of every tile in the order of
// its workgroup, where expert_of[i] is the expert of row tile i, and tile_rows
// 128 or 256.
std::vector<int64_t> moe_tile_order(std::vector<int64_t> expert_of,
                                    int64_t n_blocks, int64_t split,
                                    int64_t tile_rows) {
  using namespace moe;
  std::vector<int64_t> out;
  for (int xcd = 0; xcd < 8; ++xcd) {
    const TilePart p = tile_part_of(xcd, (int)expert_of.size(),
                                    (int)n_blocks, (int)split);
    for (int l = 0; l < (p.m1 - p.m0) * (p.n1 - p.n0); ++l) {
      int m = 0, n = 0;
      tile_of_part(
          p, tile_rows == 128 && split == 8, l,
          [&](int i) { return expert_of.at(i); },
          [&](auto f) {
            uint64_t lanes = 0;
            for (int lane = 0; lane < WAVE_SIZE; ++lane)
              lanes |= (uint64_t)f(lane) << lane;
            return lanes;
          },
          m, n);
      out.insert(out.end(), {xcd, m, n});
    }
  }
  return out;
}

// scratch: ceil(total / 2048) * num_experts ints where total > 2048, and
// 2 * num_experts more for more than 1024 experts.
void moe_align(torch::Tensor topk_ids, int64_t num_experts, int64_t tile_rows,
               torch::Tensor sorted, torch::Tensor expert_tiles,
               torch::Tensor inv_perm, torch::Tensor scratch) {
  using namespace moe;
  TORCH_CHECK(topk_ids.scalar_type() == torch::kInt32 &&
              topk_ids.is_contiguous());
  const int total = (int)topk_ids.numel();
  const int e = (int)num_experts;
  const int bm = (int)tile_rows;
  const int max_tiles = (int)expert_tiles.numel() - 1;
  TORCH_CHECK(e >= 1, "moe_align: no experts");
  TORCH_CHECK(bm >= 1 && sorted.numel() >= (int64_t)max_tiles * bm &&
              (int64_t)max_tiles * bm >=
                  total + (int64_t)std::min(e, total) * (bm - 1) - (bm - 1));
  TORCH_CHECK(inv_perm.numel() >= total);
  if (total == 0) return;
  const int blocks = ceil_div(total, ALIGN_ROWS);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const int* ids = topk_ids.data_ptr<int>();
  const int64_t parts = blocks > 1 ? (int64_t)blocks * e : 0;
  TORCH_CHECK(scratch.scalar_type() == torch::kInt32 &&
              scratch.is_contiguous() &&
              scratch.numel() >= parts + (e > LDS_EXPERTS ? 2 * e : 0));
  int* part = scratch.data_ptr<int>();
  auto launch = [&](auto in_lds) {
    constexpr bool LDS = decltype(in_lds)::value;
    if (blocks == 1) {
      hipLaunchKernelGGL(align_small_kernel<LDS>, dim3(1), dim3(THREADS), 0,
                         stream, ids, total, e, bm,
                         expert_tiles.data_ptr<int>(), max_tiles,
                         sorted.data_ptr<int>(), inv_perm.data_ptr<int>(),
                         part);
      return;
    }
    hipLaunchKernelGGL(align_count_kernel<LDS>, dim3(blocks), dim3(THREADS),
                       0, stream, ids, total, e, part);
    hipLaunchKernelGGL(align_place_kernel<LDS>, dim3(1), dim3(THREADS), 0,
                       stream, part, blocks, e, bm,
                       expert_tiles.data_ptr<int>(), max_tiles,
                       sorted.data_ptr<int>(), part + parts);
    hipLaunchKernelGGL(align_scatter_kernel<LDS>, dim3(blocks),
                       dim3(THREADS), 0, stream, ids, total, e, part,
                       sorted.data_ptr<int>(), inv_perm.data_ptr<int>());
  };
  if (e <= LDS_EXPERTS) launch(std::true_type{});
  else                  launch(std::false_type{});
  HIP_CHECK_KERNEL();
}

static void run_gemm(const torch::Tensor& a, const torch::Tensor& b,
                     int64_t b_rows, bool shuf, torch::Tensor& c,
                     const torch::Tensor& sorted,
                     const torch::Tensor& expert_tiles, int64_t topk_div,
                     int64_t total_flat, int64_t act, int64_t form) {
  using namespace moe;
  TORCH_CHECK(a.dim() == 2 && c.dim() == 2);
  TORCH_CHECK(a.is_contiguous() && b.is_contiguous() && c.is_contiguous());
  TORCH_CHECK(a.scalar_type() == b.scalar_type() &&
              a.scalar_type() == c.scalar_type());
  const int K = (int)a.size(1);
  const int N = (int)c.size(1);
  TORCH_CHECK(act >= NONE && act <= RELU2);
  TORCH_CHECK(b_rows == (act == SILU_GATED ? 2 : 1) * (int64_t)N);
  TORCH_CHECK(K % (form > 0 ? TP_K : 32) == 0 &&
                  N % (shuf ? 16 : form > 0 ? 8 : 4) == 0,
              "K must be a multiple of 32, N of 4 (tiles: 64 and 8; in "
              "fragment order N of 16)");
  const int bm = (int)moe_tile_rows(form);
  const int em = (int)c.size(0);
  const int m_tiles = em / bm;
  TORCH_CHECK(em % bm == 0 && m_tiles == (int)expert_tiles.numel() - 1 &&
              em <= sorted.numel());
  TORCH_CHECK(topk_div > 0 || a.size(0) >= em);
  if (em == 0) return;
  const bool aligned = (uintptr_t)a.data_ptr() % 16 == 0 &&
                       (uintptr_t)b.data_ptr() % 16 == 0 &&
                       a.numel() * 2 < (1ll << 32) &&
                       b_rows * K * 2 < (1ll << 32);
  const bool by_rows = form == 0 && !shuf && aligned && K % SP_K == 0;
  const int halves = act == SILU_GATED ? 2 : 1;
  const bool wide =
      (int64_t)m_tiles * ceil_div(N * halves, SR_WIDE) >= SR_FILL;
  const int cols = (form > 0  ? TL_W
                    : by_rows ? (wide ? SR_WIDE : SR_NARROW)
                              : ST_W) / halves;
  const int n_blocks = ceil_div(N, cols);
  const int split = split_of_grid(m_tiles, n_blocks);
  const int64_t blocks =
      form > 0 ? (int64_t)ceil_div(m_tiles, 8 / split) *
                     ceil_div(n_blocks, split) * 8
               : ((int64_t)m_tiles * n_blocks + 7) / 8 * 8;
  // (Tiles address rows and an expert's weights with 32 bits, and fill LDS
  // from them 16 B at a time.)
  TORCH_CHECK(form == 0 || aligned);
  TORCH_CHECK(blocks < (1ll << 30));
  auto stream = c10::hip::getCurrentHIPStream().stream();
  if (form > 0) {
    TORCH_CHECK(a.scalar_type() == torch::kBFloat16 ||
                    a.scalar_type() == torch::kHalf,
                "moe_gemm: bf16/fp16 only");
    launch_tiles({(const short*)a.data_ptr(), a.size(1),
                  (const short*)b.data_ptr(), b_rows * K,
                  (short*)c.data_ptr(), c.size(1), sorted.data_ptr<int>(),
                  expert_tiles.data_ptr<int>(), K, N, (int)topk_div,
                  (int)total_flat, m_tiles, n_blocks, split},
                 (int)form, (int)act, a.scalar_type() == torch::kBFloat16,
                 (unsigned)blocks, stream);
    HIP_CHECK_KERNEL();
    return;
  }
  dim3 grid((unsigned)blocks);
  auto launch = [&](auto tag, auto act_tag) {
    using Tag = decltype(tag);
    constexpr int ACT = decltype(act_tag)::value;
    if (by_rows) {
      auto rows = [&](auto kernel) {
        hipLaunchKernelGGL(
            kernel, grid, dim3(THREADS), 0, stream,
            (const short*)a.data_ptr(), (const short*)b.data_ptr(),
            b_rows * K, (short*)c.data_ptr(), c.size(1),
            sorted.data_ptr<int>(), expert_tiles.data_ptr<int>(), K, N,
            (int)topk_div, (int)total_flat, m_tiles, n_blocks);
      };
      if (wide) rows(moe_rows_kernel<Tag, ACT, SR_WIDE / 16>);
      else      rows(moe_rows_kernel<Tag, ACT, SR_NARROW / 16>);
      return;
    }
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(
          kernel, grid, dim3(THREADS), 0, stream,
          (const short*)a.data_ptr(),
          a.size(1), (const short*)b.data_ptr(), b_rows * K,
          (short*)c.data_ptr(), c.size(1), sorted.data_ptr<int>(),
          expert_tiles.data_ptr<int>(), K, N, (int)topk_div, (int)total_flat,
          m_tiles, n_blocks);
    };
    if (shuf) go(moe_stream_kernel<Tag, ACT, true>);
    else      go(moe_stream_kernel<Tag, ACT, false>);
  };
  auto by_act = [&](auto tag) {
    if (act == SILU_GATED)
      launch(tag, std::integral_constant<int, SILU_GATED>{});
    else if (act == RELU2)
      launch(tag, std::integral_constant<int, RELU2>{});
    else
      launch(tag, std::integral_constant<int, NONE>{});
  };
  if (a.scalar_type() == torch::kBFloat16)
    by_act(BF16Tag{});
  else if (a.scalar_type() == torch::kHalf)
    by_act(FP16Tag{});
  else
    TORCH_CHECK(false, "moe_gemm: bf16/fp16 only");
  HIP_CHECK_KERNEL();
}

// c [EM, N] = act(a rows x b[expert]^T); b [E, N, K], or [E, 2N, K] for the
// gated activation. topk_div > 0: a's rows are tokens, gathered through
// `sorted`; 0: a's rows are in tile order already.
void moe_gemm(torch::Tensor a, torch::Tensor b, torch::Tensor c,
              torch::Tensor sorted, torch::Tensor expert_tiles,
              int64_t topk_div, int64_t total_flat, int64_t act,
              int64_t form) {
  TORCH_CHECK(b.dim() == 3 && b.size(2) == a.size(1), "B inner dim mismatch");
  run_gemm(a, b, b.size(1), false, c, sorted, expert_tiles, topk_div,
           total_flat, act, form);
}

// The same with b in fragment order, [E, n * k].
void moe_gemm_shuf(torch::Tensor a, torch::Tensor b_shuf, torch::Tensor c,
                   torch::Tensor sorted, torch::Tensor expert_tiles,
                   int64_t n, int64_t k, int64_t topk_div,
                   int64_t total_flat, int64_t act) {
  TORCH_CHECK(a.size(1) == k && b_shuf.numel() % (n * k) == 0);
  run_gemm(a, b_shuf, n, true, c, sorted, expert_tiles, topk_div, total_flat,
           act, 0);
}

void moe_combine(torch::Tensor out, torch::Tensor y,
                 torch::Tensor topk_weights, torch::Tensor inv_perm) {
  using namespace moe;
  TORCH_CHECK(out.dim() == 2 && y.dim() == 2);
  TORCH_CHECK(out.is_contiguous() && y.is_contiguous());
  TORCH_CHECK(topk_weights.scalar_type() == torch::kFloat);
  const int T = (int)out.size(0);
  const int H = (int)out.size(1);
  const int topk = (int)topk_weights.size(1);
  TORCH_CHECK(H % 8 == 0);
  TORCH_CHECK(y.size(1) == H);
  const int parts = ceil_div(H, COMBINE * 8);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto launch = [&](auto tag) {
    using Tag = decltype(tag);
    const bool once = (int64_t)T * topk * H * 2 >= READ_ONCE_BYTES;
    hipLaunchKernelGGL((once ? combine_kernel<Tag, true>
                             : combine_kernel<Tag, false>),
                       dim3(T * parts), dim3(COMBINE), 0, stream,
                       (short*)out.data_ptr(), (const short*)y.data_ptr(),
                       y.size(1), topk_weights.data_ptr<float>(),
                       inv_perm.data_ptr<int>(), topk, H, parts);
  };
  if (out.scalar_type() == torch::kBFloat16)
    launch(BF16Tag{});
  else if (out.scalar_type() == torch::kHalf)
    launch(FP16Tag{});
  else
    TORCH_CHECK(false, "moe_combine: bf16/fp16 only");
  HIP_CHECK_KERNEL();
}


}  // namespace vllm_amd
