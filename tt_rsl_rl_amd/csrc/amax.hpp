// Largest magnitudes of tensors, as the kernels that write them leave them and the fp16x3 GEMMs read them.
#pragma once

#include "common.hpp"

namespace ppo {
namespace {

constexpr int kAmaxSlots = PPO_AMAX_SLOTS;
constexpr int kAmaxStride = PPO_AMAX_WORDS / PPO_AMAX_SLOTS;  // a line per slot: atomics on one line serialise
static_assert(kAmaxSlots == 64, "one slot per lane");

// Largest value over the wave, in every lane (DPP rotations within 16 lanes, then the four rows through scalar registers: no LDS
// round trip on the kernel's first loads).
__device__ __forceinline__ uint32_t wave_max(uint32_t u) {
  u = max(u, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(u), 0x121, 0xf, 0xf, false)));
  u = max(u, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(u), 0x122, 0xf, 0xf, false)));
  u = max(u, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(u), 0x124, 0xf, 0xf, false)));
  u = max(u, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(u), 0x128, 0xf, 0xf, false)));
  const uint32_t a = __builtin_amdgcn_readlane(u, 0), b = __builtin_amdgcn_readlane(u, 16),
                 c = __builtin_amdgcn_readlane(u, 32), d = __builtin_amdgcn_readlane(u, 48);
  return max(max(a, b), max(c, d));
}

// The power of two that brings a tensor's largest magnitude (fp32 bits u) into [2^14, 2^15), as its exponent.  Zero
// (an all-zero tensor) gives 0; a non-finite or tiny largest value the closest exponent that keeps 2^e and 2^-e normal.
__device__ __forceinline__ int amax_exponent(uint32_t u) {
  if (u == 0) return 0;
  return min(max(141 - static_cast<int>(u >> 23), -113), 126);
}
__device__ __forceinline__ float pow2(int e) { return __builtin_bit_cast(float, static_cast<uint32_t>(e + 127) << 23); }

// The wave's largest magnitude into the tensor's slots.
__device__ __forceinline__ void amax_publish(uint32_t* slots, float m, int lane, int slot) {
  const uint32_t u = wave_max(__builtin_bit_cast(uint32_t, m));
  if (lane == 0) atomicMax(slots + (slot & (kAmaxSlots - 1)) * kAmaxStride, u);
}


// m = max(m, |a|, |b|); a NaN does not count.
__device__ __forceinline__ void raise2(float& m, float a, float b) {
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a), "v"(b));
}

}  // namespace
}  // namespace ppo
