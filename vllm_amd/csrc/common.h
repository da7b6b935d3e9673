// Common device helpers for vllm_amd CDNA4 (gfx950) kernels.
//
// Written for MI355X only: wave64, 64-bank LDS, MFMA matrix cores,
// HBM3E. No CUDA-compat paths.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <cstdint>
#include <type_traits>
#include <utility>

#define WAVE_SIZE 64

#define DEVINL __device__ __forceinline__

// ---------------------------------------------------------------------------
// Vector types for wide loads (G13: always vectorize bf16 loads).
typedef short  s16x8 __attribute__((ext_vector_type(8)));   // 8 bf16 = 16B
typedef short  s16x4 __attribute__((ext_vector_type(4)));   // 8B
typedef float  f32x4 __attribute__((ext_vector_type(4)));
typedef float  f32x2 __attribute__((ext_vector_type(2)));
typedef float  f32x16 __attribute__((ext_vector_type(16)));
typedef int    i32x4 __attribute__((ext_vector_type(4)));

// MFMA fragment types (gfx950 16x16x32 bf16: A/B = 8 bf16, C/D = 4 f32).
typedef s16x8 frag_b16;
typedef f32x4 frag_f32;

DEVINL float bf16_to_f32(short v) {
  union {
    float f;
    uint32_t u;
  } cvt;
  cvt.u = (uint32_t)(uint16_t)v << 16;
  return cvt.f;
}

DEVINL short f32_to_bf16(float f) {
  union {
    float f;
    uint32_t u;
  } cvt;
  cvt.f = f;
  // round-to-nearest-even
  uint32_t lsb = (cvt.u >> 16) & 1;
  uint32_t rounded = cvt.u + 0x7fffu + lsb;
  return (short)(rounded >> 16);
}

DEVINL float f16_to_f32(short v) { return __half2float(__ushort_as_half((uint16_t)v)); }
DEVINL short f16_from_f32(float f) { return (short)__half_as_ushort(__float2half(f)); }

// Generic scalar converters selected by template tag.
struct BF16Tag {};
struct FP16Tag {};

template <typename Tag> DEVINL float to_f32(short v);
template <> DEVINL float to_f32<BF16Tag>(short v) { return bf16_to_f32(v); }
template <> DEVINL float to_f32<FP16Tag>(short v) { return f16_to_f32(v); }

template <typename Tag> DEVINL short from_f32(float f);
template <> DEVINL short from_f32<BF16Tag>(float f) { return f32_to_bf16(f); }
template <> DEVINL short from_f32<FP16Tag>(float f) { return f16_from_f32(f); }

// ---------------------------------------------------------------------------
// OCP fp8 e4m3fn (bias 7, no inf, 0x7f/0xff = NaN, max finite 448) — the
// gfx950-native FP8 format and torch.float8_e4m3fn. Used for the fp8 KV
// cache (kv_cache_dtype="fp8"): halves attention HBM traffic and doubles
// KV capacity.
// gfx950 has single-instruction OCP fp8 converts (v_cvt_f32_fp8 /
// v_cvt_pk_fp8_f32, RNE) — the software bit manipulation this replaced
// cost ~20 VALU ops per element and made the fp8-KV decode kernel
// conversion-bound instead of HBM-bound.
DEVINL uint8_t f32_to_fp8_e4m3(float f) {
  union { float f; uint32_t u; } c;
  c.f = f;
  // Saturate finite values to +-448 (max finite e4m3); NaN propagates
  // through the hardware convert (same recipe as amd_hip_fp8.h).
  float cl = f;
  if ((c.u & 0x7F800000u) != 0x7F800000u)
    cl = __builtin_amdgcn_fmed3f(f, 448.f, -448.f);
  return (uint8_t)__builtin_amdgcn_cvt_pk_fp8_f32(cl, cl, 0, false);
}

// Cache element traits: the KV cache may be narrower than the compute
// dtype. vec8 loads 8 cache elements (16 B bf16/fp16, 8 B fp8).
typedef uint8_t u8x8 __attribute__((ext_vector_type(8)));
struct FP8CacheTag {};

template <typename CTag> struct CacheTraits;
template <> struct CacheTraits<BF16Tag> {
  using elem = short;
  using vec8 = s16x8;
  static DEVINL elem put(float f) { return f32_to_bf16(f); }
};
template <> struct CacheTraits<FP16Tag> {
  using elem = short;
  using vec8 = s16x8;
  static DEVINL elem put(float f) { return f16_from_f32(f); }
};
template <> struct CacheTraits<FP8CacheTag> {
  using elem = uint8_t;
  using vec8 = u8x8;
  static DEVINL elem put(float f) { return f32_to_fp8_e4m3(f); }
};

// ---------------------------------------------------------------------------
// Matrix-core helpers. The 16-bit element type selects the instruction:
// bf16 and fp16 bits share the fragment registers (s16x8), so a kernel
// templated on the tag must go through these rather than name one
// builtin.
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));

template <typename Tag> DEVINL f32x4 mfma16(s16x8 a, s16x8 b, f32x4 c);
template <> DEVINL f32x4 mfma16<BF16Tag>(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(b16x8, a), __builtin_bit_cast(b16x8, b), c, 0, 0, 0);
}
template <> DEVINL f32x4 mfma16<FP16Tag>(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(
      __builtin_bit_cast(h16x8, a), __builtin_bit_cast(h16x8, b), c, 0, 0, 0);
}
// The same over 16 instead of 32.
template <typename Tag> DEVINL f32x4 mfma16(s16x4 a, s16x4 b, f32x4 c);
template <> DEVINL f32x4 mfma16<BF16Tag>(s16x4 a, s16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
template <> DEVINL f32x4 mfma16<FP16Tag>(s16x4 a, s16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(
      __builtin_bit_cast(h16x4, a), __builtin_bit_cast(h16x4, b), c, 0, 0, 0);
}
template <typename Tag> DEVINL f32x16 mfma32(s16x8 a, s16x8 b, f32x16 c);
template <> DEVINL f32x16 mfma32<BF16Tag>(s16x8 a, s16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
      __builtin_bit_cast(b16x8, a), __builtin_bit_cast(b16x8, b), c, 0, 0, 0);
}
template <> DEVINL f32x16 mfma32<FP16Tag>(s16x8 a, s16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(
      __builtin_bit_cast(h16x8, a), __builtin_bit_cast(h16x8, b), c, 0, 0, 0);
}

// c += a b, 16 x 16 x 32, c in accumulation registers and in its place. The
// builtin names result and sum apart: where all 256 accumulation registers
// are taken the compiler then moves them about (8192 x 28672 x 4096 by
// tile_product.h 1.08 PFLOP/s, 1.43 so). The compiler knows nothing of
// what may stand right before and after the instruction, so accumulators come
// and go through acc_fence; that nothing else was put beside one is checked in
// the built kernels (tests/test_product_waits.py).
template <typename Tag> DEVINL void mfma16_acc(f32x4& c, s16x8 a, s16x8 b) {
  if constexpr (std::is_same_v<Tag, BF16Tag>)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                 : "+a"(c)
                 : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0"
                 : "+a"(c)
                 : "v"(a), "v"(b));
}
// Between other instructions that write or read the accumulators and products
// that do: the waits of either side (two states before a product, eight after)
// lie before and behind the point where the compiler may move them.
template <int N, int M> DEVINL void acc_fence(f32x4 (&acc)[N][M]) {
  asm volatile("s_nop 15");
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) asm volatile("" : "+a"(acc[i][j]));
  asm volatile("s_nop 15");
}

// f(0) to f(N - 1), each with its number as a constant. (Unrolled loops stay
// loops where their bodies are long, and arrays of registers then go to
// scratch.)
template <int N, typename F, int... I>
DEVINL void unrolled(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> DEVINL void unrolled(F f) {
  unrolled<N>(f, std::make_integer_sequence<int, N>{});
}

// Two floats rounded (nearest even) to a packed 16-bit pair.
template <typename Tag> DEVINL int pack2(float a, float b);
template <> DEVINL int pack2<BF16Tag>(float a, float b) {
  return __builtin_bit_cast(
      int, __builtin_convertvector((f32x2){a, b}, b16x2));
}
template <> DEVINL int pack2<FP16Tag>(float a, float b) {
  return __builtin_bit_cast(
      int, __builtin_convertvector((f32x2){a, b}, h16x2));
}
template <typename Tag> DEVINL float unpack_lo(int v) {
  return to_f32<Tag>((short)v);
}
template <typename Tag> DEVINL float unpack_hi(int v) {
  return to_f32<Tag>((short)(v >> 16));
}

// acc plus the two values of a packed pair, in fp32.
template <typename Tag> DEVINL float add_pair(int v, float acc);
template <> DEVINL float add_pair<BF16Tag>(int v, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(
      __builtin_bit_cast(b16x2, v), __builtin_bit_cast(b16x2, 0x3f803f80),
      acc, false);
}
template <> DEVINL float add_pair<FP16Tag>(int v, float acc) {
  return __builtin_amdgcn_fdot2(
      __builtin_bit_cast(h16x2, v), __builtin_bit_cast(h16x2, 0x3c003c00),
      acc, false);
}

// Four e4m3 bytes to four 16-bit values (exact for both types).
template <typename Tag> DEVINL int2 fp8x4_widen(int v);
template <> DEVINL int2 fp8x4_widen<BF16Tag>(int v) {
  return {__builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                      v, 1.0f, false)),
          __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                      v, 1.0f, true))};
}
template <> DEVINL int2 fp8x4_widen<FP16Tag>(int v) {
  return {__builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(
                                      v, 1.0f, false)),
          __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(
                                      v, 1.0f, true))};
}

// Column l32 of a 32 x 32 product holds rows 8*b + 4*half + 0..3 in
// registers 4*b ..; the lower half wave receives all eight rows of b, the
// upper one those of b + 1: one 16 B store a lane, 32 B in a row (8 B
// stores: 30 % slower where a kernel is bound by what it writes).
template <typename Tag> DEVINL i32x4 row_chunk(const f32x16& c, int b) {
  const unsigned x0 = pack2<Tag>(c[b * 4], c[b * 4 + 1]);
  const unsigned x1 = pack2<Tag>(c[b * 4 + 2], c[b * 4 + 3]);
  const unsigned y0 = pack2<Tag>(c[b * 4 + 4], c[b * 4 + 5]);
  const unsigned y1 = pack2<Tag>(c[b * 4 + 6], c[b * 4 + 7]);
  const auto s0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
  const auto s1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
  const int a0 = s0[0], a1 = s1[0], b0 = s0[1], b1 = s1[1];
  return i32x4{a0, a1, b0, b1};
}

// The same of two 16 x 16 products with the columns of 16 x 16 in a row: lane
// l16 of group l4 holds rows 4 * l4 + 0..3 of each, and gets eight rows from
// row_start16() of the pair's 32 on.
DEVINL int row_start16() {
  const int l4 = threadIdx.x % WAVE_SIZE >> 4;
  return (l4 & 1) * 16 + (l4 >> 1) * 8;
}
template <typename Tag> DEVINL i32x4 row_chunk16(f32x4 a, f32x4 b) {
  const auto s0 = __builtin_amdgcn_permlane16_swap(
      pack2<Tag>(a[0], a[1]), pack2<Tag>(b[0], b[1]), false, false);
  const auto s1 = __builtin_amdgcn_permlane16_swap(
      pack2<Tag>(a[2], a[3]), pack2<Tag>(b[2], b[3]), false, false);
  const int a0 = s0[0], a1 = s1[0], b0 = s0[1], b1 = s1[1];
  return i32x4{a0, a1, b0, b1};
}

// Rotates 8 pairs (x1[j], x2[j]) by the angles p0 + j of a table row
// [cos(half) | sin(half)].
template <typename Tag>
DEVINL void rope8(s16x8& x1, s16x8& x2, const float* __restrict__ cs,
                  int half, int p0) {
  f32x4 c[2], s[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    c[i] = *reinterpret_cast<const f32x4*>(cs + p0 + i * 4);
    s[i] = *reinterpret_cast<const f32x4*>(cs + half + p0 + i * 4);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float a = to_f32<Tag>(x1[j]), b = to_f32<Tag>(x2[j]);
    const float cj = c[j >> 2][j & 3], sj = s[j >> 2][j & 3];
    x1[j] = from_f32<Tag>(__builtin_fmaf(a, cj, -(b * sj)));
    x2[j] = from_f32<Tag>(__builtin_fmaf(a, sj, b * cj));
  }
}

// Transposing LDS read: the 16 lanes of a group address a block of 4
// rows x 16 columns of 16-bit values (lane i: row i / 4, columns
// (i % 4) * 4 .. + 3) and lane i receives column i, rows 0..3.
DEVINL s16x4 lds_read_tr(const void* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)p);
}

// Order for the scheduler, said after STEPS steps of LDS reads and MFMAS
// products each: AHEAD reads come first, then PER further ones after each
// step. By itself it tends to wait for every read just before its product
// where registers are short.
template <int AHEAD, int PER, int STEPS, int MFMAS = 1>
DEVINL void reads_ahead() {
  __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, MFMAS, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);
  }
}

// 16 B from global memory; ONCE: a line that nobody reads again, which
// leaves the caches first.
template <bool ONCE> DEVINL s16x8 load16(const short* p) {
  const s16x8* v = reinterpret_cast<const s16x8*>(p);
  return ONCE ? __builtin_nontemporal_load(v) : *v;
}

// A value that no lane's place decides and that the launch does not change:
// by way of the scalar cache. (A pointer that comes in a structure is not
// known to be free of aliases. The compiler then loads through it as a vector,
// and such a load waits for all that were issued before it.)
DEVINL int load_uniform(const int* p) {
  return *(const __attribute__((address_space(4))) int*)p;
}

// 64 lanes x 16 B from global memory straight into LDS: lane i's 16 bytes
// land at dst + 16 * i (dst the same in all lanes). No register receives
// anything, so the kernel waits itself (lds_fill_wait, then a barrier for
// the other waves' parts): the compiler would wait for every fill under
// way before each LDS read, having no means to tell the tiles apart.
DEVINL void lds_fill16(const void* src, void* dst) {
  const uint32_t at = (uint32_t)(uintptr_t)(
      __attribute__((address_space(3))) void*)dst;
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(at), "v"(src)
      : "memory", "m0");
}
// The same from base + at, base the same in all lanes.
DEVINL void lds_fill16(const void* base, uint32_t at, void* dst) {
  const uint32_t to = (uint32_t)(uintptr_t)(
      __attribute__((address_space(3))) void*)dst;
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(to), "v"(at), "s"(base)
      : "memory", "m0");
}
// The same for what is read once: its lines are the first to leave L2, what
// is read again stays (8 rows of 28672 x 4096: 43.0 us with plain fills of
// the weights, 39.3 so).
DEVINL void lds_fill16_once(const void* base, uint32_t at, void* dst) {
  const uint32_t to = (uint32_t)(uintptr_t)(
      __attribute__((address_space(3))) void*)dst;
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2 nt"
      :
      : "s"(to), "v"(at), "s"(base)
      : "memory", "m0");
}
// mfma16_acc and, behind it, a fill of the 16 * 64 bytes `off` after `to` (an
// address in LDS; off a constant). The place goes to m0 before the product, so
// that the wait between the two holds the product, and the next product does
// not wait for the instructions of a fill of its own.
template <bool ONCE, typename Tag>
DEVINL void mfma16_acc_fill(f32x4& c, s16x8 a, s16x8 b, const void* base,
                            uint32_t at, uint32_t to, int off) {
#define VLLM_AMD_PRODUCT_FILL(TYPE, HINT)                          \
  asm volatile("s_add_u32 m0, %3, %4\n\t"                          \
               "v_mfma_f32_16x16x32_" TYPE " %0, %1, %2, %0\n\t"   \
               "global_load_lds_dwordx4 %5, %6" HINT               \
               : "+a"(c)                                           \
               : "v"(a), "v"(b), "s"(to), "i"(off), "v"(at), "s"(base) \
               : "memory", "m0", "scc")
  constexpr bool BF16 = std::is_same_v<Tag, BF16Tag>;
  if constexpr (BF16 && ONCE)      VLLM_AMD_PRODUCT_FILL("bf16", " nt");
  else if constexpr (BF16)         VLLM_AMD_PRODUCT_FILL("bf16", "");
  else if constexpr (ONCE)         VLLM_AMD_PRODUCT_FILL("f16", " nt");
  else                             VLLM_AMD_PRODUCT_FILL("f16", "");
#undef VLLM_AMD_PRODUCT_FILL
}
// At most N (< 64) of this wave's loads still under way; the builtin, so
// that the compiler knows its own older loads to be done as well and does
// not wait again after the next fill.
template <int N = 0> DEVINL void lds_fill_wait() {
  static_assert(N >= 0 && N < 64);
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}
// All of this wave's LDS operations, or all of its loads and stores, are done.
// The builtin says nothing of memory to the compiler: without a barrier on
// either side an access might be moved past the wait that is meant for it.
DEVINL void lds_wait() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
  asm volatile("" ::: "memory");
}
DEVINL void global_wait() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
  asm volatile("" ::: "memory");
}
// Workgroup barrier that waits for this wave's LDS operations but not for
// its loads (__syncthreads may wait for both).
DEVINL void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ---------------------------------------------------------------------------
// Wave reductions (64 lanes).
DEVINL float wave_reduce_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

DEVINL float wave_reduce_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// The value of the lane N before this one in its group of 16, round it.
template <int N> DEVINL float row_ror(float v) {
  const int b = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(b, b, 0x120 + N, 0xf, 0xf, false));
}

// Reduce within 16-lane groups (used for MFMA row reductions).
DEVINL float group16_reduce_max(float v) {
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

DEVINL float group16_reduce_sum(float v) {
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Block reduction via LDS (block size must be multiple of 64).
template <int MAX_WAVES>
DEVINL float block_reduce_sum(float v, float* lds_scratch) {
  const int wave = threadIdx.x / WAVE_SIZE;
  const int lane = threadIdx.x % WAVE_SIZE;
  const int nwaves = blockDim.x / WAVE_SIZE;
  v = wave_reduce_sum(v);
  if (lane == 0) lds_scratch[wave] = v;
  __syncthreads();
  float r = (lane < nwaves) ? lds_scratch[lane] : 0.f;
#pragma unroll
  for (int off = MAX_WAVES / 2; off > 0; off >>= 1)
    r += __shfl_xor(r, off, 64);
  return __shfl(r, 0, 64);
}

// ---------------------------------------------------------------------------
#define HIP_CHECK_KERNEL()                                    \
  do {                                                        \
    hipError_t e = hipGetLastError();                         \
    if (e != hipSuccess) {                                    \
      TORCH_CHECK(false, "HIP kernel launch failed: ",        \
                  hipGetErrorString(e));                      \
    }                                                         \
  } while (0)

DEVINL int ceil_div_dev(int a, int b) { return (a + b - 1) / b; }
inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
