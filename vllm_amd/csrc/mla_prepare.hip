// What stands between the projections of an MLA block and its attention,
// in one pass (gfx950): the latent is normalized and written to the paged
// cache with its rotated key part, the queries' rotary parts are rotated
// into a tensor of their own.
//
// Few tokens: bound by launches (ten small ones before: slices copied,
// norm, rotation, two indexed writes and their indices), many: by memory,
// 2 x 16 KB of query parts a token at 128 heads. One workgroup a token:
// four waves take the query heads, 16 B a lane from each half of a head, a
// fifth the latent row (512 values, 8 a lane) and the key part, so the
// norm's reduction stays in a wave. 128 heads, us: 128 tokens 44 -> 4.4;
// 3901 tokens 105 -> 27 (4.9 TB/s).

#include <torch/all.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include "common.h"

namespace vllm_amd {

namespace {

constexpr int LORA = 512;
constexpr int ROPE = 64;
constexpr int Q_THREADS = 4 * WAVE_SIZE;
constexpr int THREADS = Q_THREADS + WAVE_SIZE;

template <typename Tag>
__launch_bounds__(THREADS) __global__
void mla_prepare_kernel(short* __restrict__ q_out,        // [T, H, ROPE]
                        short* __restrict__ cache,        // [slots, 576]
                        const short* __restrict__ q, int64_t q_row,
                        int64_t q_head, const short* __restrict__ kv,
                        int64_t kv_row,                   // [T, LORA + ROPE]
                        const short* __restrict__ weight, float eps,
                        const float* __restrict__ cos_sin,
                        const int64_t* __restrict__ positions,
                        const int64_t* __restrict__ slots, int heads) {
  const int64_t t = blockIdx.x;
  const float* cs = cos_sin + positions[t] * ROPE;
  if (threadIdx.x < Q_THREADS) {
    for (int i = threadIdx.x; i < heads * 4; i += Q_THREADS) {
      const int h = i >> 2, p0 = (i & 3) * 8;
      const short* src = q + t * q_row + h * q_head + p0;
      s16x8 x1 = *reinterpret_cast<const s16x8*>(src);
      s16x8 x2 = *reinterpret_cast<const s16x8*>(src + ROPE / 2);
      rope8<Tag>(x1, x2, cs, ROPE / 2, p0);
      short* dst = q_out + (t * heads + h) * ROPE + p0;
      *reinterpret_cast<s16x8*>(dst) = x1;
      *reinterpret_cast<s16x8*>(dst + ROPE / 2) = x2;
    }
    return;
  }
  const int64_t slot = slots[t];
  if (slot < 0) return;   // padding
  const int lane = threadIdx.x - Q_THREADS;
  const short* row = kv + t * kv_row;
  short* dst = cache + slot * (LORA + ROPE);
  s16x8 v = *reinterpret_cast<const s16x8*>(row + lane * 8);
  const s16x8 w = *reinterpret_cast<const s16x8*>(weight + lane * 8);
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float f = to_f32<Tag>(v[j]);
    ss += f * f;
  }
  const float inv = rsqrtf(wave_reduce_sum(ss) / LORA + eps);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = from_f32<Tag>(to_f32<Tag>(v[j]) * inv * to_f32<Tag>(w[j]));
  *reinterpret_cast<s16x8*>(dst + lane * 8) = v;
  if (lane < 4) {
    const short* src = row + LORA + lane * 8;
    s16x8 x1 = *reinterpret_cast<const s16x8*>(src);
    s16x8 x2 = *reinterpret_cast<const s16x8*>(src + ROPE / 2);
    rope8<Tag>(x1, x2, cs, ROPE / 2, lane * 8);
    *reinterpret_cast<s16x8*>(dst + LORA + lane * 8) = x1;
    *reinterpret_cast<s16x8*>(dst + LORA + ROPE / 2 + lane * 8) = x2;
  }
}

}  // namespace

// q_pe [T, H, 64] (strided) -> its rotation, contiguous; kv_a [T, 576] ->
// normalized latent and rotated key part in the cache's slots.
torch::Tensor mla_prepare(torch::Tensor positions, torch::Tensor q_pe,
                          torch::Tensor kv_a, torch::Tensor weight,
                          double eps, torch::Tensor cos_sin,
                          torch::Tensor kv_cache, torch::Tensor slots) {
  TORCH_CHECK(q_pe.dim() == 3 && q_pe.size(2) == ROPE && kv_a.dim() == 2 &&
              kv_a.size(1) == LORA + ROPE && weight.numel() == LORA &&
              kv_cache.dim() == 3 && kv_cache.size(2) == LORA + ROPE,
              "mla_prepare: latent of 512 + 64");
  const int64_t T = q_pe.size(0);
  TORCH_CHECK(kv_a.size(0) == T && positions.numel() == T &&
              slots.numel() == T);
  const auto type = q_pe.scalar_type();
  TORCH_CHECK((type == torch::kBFloat16 || type == torch::kHalf) &&
              kv_a.scalar_type() == type && weight.scalar_type() == type &&
              kv_cache.scalar_type() == type);
  auto rows_ok = [](const torch::Tensor& x) {
    bool ok = x.stride(-1) == 1 && (uintptr_t)x.data_ptr() % 16 == 0;
    for (int64_t d = 0; d + 1 < x.dim(); ++d) ok &= x.stride(d) % 8 == 0;
    return ok;
  };
  TORCH_CHECK(rows_ok(q_pe) && rows_ok(kv_a) && weight.is_contiguous() &&
              rows_ok(weight) && kv_cache.is_contiguous() &&
              positions.is_contiguous() && slots.is_contiguous(),
              "mla_prepare: rows must be 16 B aligned");
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 &&
              cos_sin.is_contiguous() && cos_sin.size(-1) == ROPE);
  auto out = torch::empty({T, q_pe.size(1), ROPE}, q_pe.options());
  if (T == 0) return out;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto launch = [&](auto tag) {
    using Tag = decltype(tag);
    hipLaunchKernelGGL(
        (mla_prepare_kernel<Tag>), dim3(T), dim3(THREADS), 0, stream,
        (short*)out.data_ptr(), (short*)kv_cache.data_ptr(),
        (const short*)q_pe.data_ptr(), q_pe.stride(0), q_pe.stride(1),
        (const short*)kv_a.data_ptr(), kv_a.stride(0),
        (const short*)weight.data_ptr(), (float)eps,
        cos_sin.data_ptr<float>(), positions.data_ptr<int64_t>(),
        slots.data_ptr<int64_t>(), (int)q_pe.size(1));
  };
  if (type == torch::kBFloat16) launch(BF16Tag{});
  else launch(FP16Tag{});
  HIP_CHECK_KERNEL();
  return out;
}

}  // namespace vllm_amd
