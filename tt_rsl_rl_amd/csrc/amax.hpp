// Ranges of tensors, as the kernels that write them leave them and the fp16x3 GEMMs read them.  A slot's first word is the
// largest magnitude (fp32 bits), its second the smallest among the nonzero largest magnitudes of the tensor's parts, as
// part_code() of it (0: no such part).
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

// The second word for a part whose largest magnitude has the bits u: larger for a smaller part (an atomic maximum finds the
// smallest), and as a float negative, so that the words' largest float is the first word's.
__device__ __forceinline__ uint32_t part_code(uint32_t u) { return u == 0 ? 0u : 0x80000000u | (0x7f800000u - u); }

// A tensor as fp16x3 operand.  Scaled by its largest magnitude, an element is held to 2^-50 of that, so one part far above
// the others (a sentinel in one row, a column of another unit) would cost the others their digits: to 2^-22 of a part 2^28
// below the largest, whence kMaxSpread.  The parts of the inputs and the weights are single rows and columns, those of
// activations and gradients the tiles of the waves that write them (16 to 64 rows): an outlier there comes of one in the
// inputs or the weights, which amax_publish hands on, or of single rows of the loss.  Not seen are rows and columns of
// gradients that are small in every tile, such as those of a unit that ELU saturates in every row (at z = -25 they are
// 2^-36 of the others' and kept to 2^-14 of themselves): their sums matter to that unit alone, whose steps they leave as
// they are (Adam divides by no less than its eps of 1e-8, which gradients clipped to a norm of 1 are far below there).
// Operands beyond the spread, with an infinity, or so large (2^61) that the two scales taken out one after the other could
// overflow in between, are multiplied in three bf16 parts, which have fp32's exponents.
constexpr int kMaxSpread = 28, kMaxExponent = 127 + 60;
struct Range {
  uint32_t top, low;
  __device__ __forceinline__ bool narrow() const {
    const int smallest = low == 0 ? 255 : static_cast<int>((0x7f800000u - (low & 0x7fffffffu)) >> 23);
    return static_cast<int>(top >> 23) <= kMaxExponent && static_cast<int>(top >> 23) - smallest <= kMaxSpread;
  }
};
__device__ __forceinline__ Range load_range(const uint32_t* slots, int lane) {
  const uint2 u = *reinterpret_cast<const uint2*>(slots + lane * kAmaxStride);
  return Range{wave_max(u.x), wave_max(u.y)};
}

// A wave's range into the tensor's slots.
__device__ __forceinline__ void publish_range(uint32_t* slots, uint32_t top, uint32_t low, int lane, int slot) {
  if (lane != 0 || top == 0) return;
  uint32_t* const w = slots + (slot & (kAmaxSlots - 1)) * kAmaxStride;
  atomicMax(w, top);
  atomicMax(w + 1, low);
}

// The same where the wave's values are one part.  wide: the tensor comes of one that is not narrow, so that outliers may lie
// in every part: it counts as not narrow itself, and so does what follows from it.
constexpr uint32_t kWideCode = 0x80000000u | (0x7f800000u - 1u);
__device__ __forceinline__ void amax_publish(uint32_t* slots, float m, bool wide, int lane, int slot) {
  const uint32_t u = wave_max(__builtin_bit_cast(uint32_t, m));
  publish_range(slots, u, wide ? kWideCode : part_code(u), lane, slot);
}
__device__ __forceinline__ bool wide_source(const uint32_t* slots, int lane) {
  return slots != nullptr && !load_range(slots, lane).narrow();
}

// m = max(m, |a|, |b|); a NaN does not count.
__device__ __forceinline__ void raise2(float& m, float a, float b) {
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a), "v"(b));
}

}  // namespace
}  // namespace ppo
