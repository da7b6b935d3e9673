// Sums and partial results that meet in the last workgroup of a group to
// arrive (gfx950): the others write their parts and leave, nobody waits.
//
// Workgroups of a group run on different XCDs, whose L2s do not see each
// other. Parts are written and read by agent-scope accesses, which go past
// them; a release fence instead would write back all of L2 (2112 x 7168, 64
// rows in three parts: 33 us with fences, 14.3 without).
#pragma once

#include "common.h"

namespace at {
class Tensor;
}

namespace vllm_amd {

// Zeroed counters 0 .. n - 1 for a launch on the current stream of like's
// device; the launch leaves them zero. (bindings of torch: arrivals.cpp)
at::Tensor arrival_counters(const at::Tensor& like, int64_t n);

// Where counter i lies. Arrivals at one line of 128 B are served one after the
// other, and all workgroups of a launch may end at once, so neighbours lie on
// different lines: 512 of them, again and again, in blocks of ARRIVAL_BLOCK
// counters (1 row x 8000 keys, 8 KV heads: 15.1 us side by side, 13.2 so).
constexpr int ARRIVAL_BLOCK = 16384;
inline __host__ __device__ int64_t arrival_place(int64_t i) {
  return (i & ~(int64_t)(ARRIVAL_BLOCK - 1)) + (i & 511) * 32 +
         ((i >> 9) & 31);
}

DEVINL void part_put(f32x4* p, f32x4 v) {
  const i32x4 b = __builtin_bit_cast(i32x4, v);
  uint64_t* q = reinterpret_cast<uint64_t*>(p);
  __hip_atomic_store(q, (uint64_t)(uint32_t)b[0] | (uint64_t)b[1] << 32,
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(q + 1, (uint64_t)(uint32_t)b[2] | (uint64_t)b[3] << 32,
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL f32x4 part_get(const f32x4* p) {
  const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
  const uint64_t a =
      __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint64_t b =
      __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __builtin_bit_cast(
      f32x4, (i32x4){(int)a, (int)(a >> 32), (int)b, (int)(b >> 32)});
}
DEVINL void part_put(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL float part_get(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Called by all threads of a workgroup after its part_puts; true in the
// last of `total` workgroups that come to counter i, which may then
// part_get what all have put. `flag` is a word of LDS that nothing else
// uses until the next barrier.
DEVINL bool last_to_arrive(unsigned* counters, int64_t i, unsigned total,
                           unsigned* flag) {
  // Every wave's parts are written through before the workgroup counts.
  global_wait();
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned* counter = counters + arrival_place(i);
    const unsigned before = __hip_atomic_fetch_add(
        counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = before == total - 1;
    if (last)   // zero again for the next launch
      __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  const bool last = *flag != 0;
  asm volatile("" ::: "memory");
  return last;
}

}  // namespace vllm_amd
