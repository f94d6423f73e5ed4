// The bound that the wavefronts of a sampled draw share (row_sample_kernel): log2 of a key, as a float whose bits are compared as
// an unsigned integer.  2^23 (log2(key) - 23 + 256): positive for every fp32 key above zero, so that larger keys have larger bits.
#pragma once
#include <hip/hip_runtime.h>

namespace subspec {

constexpr float kSeenBias = 256.0f * 0x1p23f;

// bits of a positive key, from below (1.5e-4 covers the roundings).  The logarithm comes in front of the scaling: a key below 2^-127
// would not survive the product, and the bits of -inf are more than any real bound has -- such a slice would evaluate every element
// to its end.
__host__ __device__ inline uint32_t seen_bits_of(float key) {
  const float bits = (log2f(key) - (23.0f + 1.5e-4f)) * 0x1p23f + kSeenBias;
  return __builtin_bit_cast(uint32_t, bits);
}
// Bits that the row's drawn key reaches whatever its words are: its largest element, of probability `pmax`, has a key of at least
// pmax / -log(2^-24) = pmax / 16.64.  0 (no bound) for a row whose probabilities are all zero or NaN.
__host__ __device__ inline uint32_t least_seen_bits(float pmax) { return pmax > 0.f ? seen_bits_of(0.06f * pmax) : 0u; }
// 2^23 (log2(key) - 23) again
__host__ __device__ inline float seen_level(uint32_t bits) { return __builtin_bit_cast(float, bits) - kSeenBias; }

}  // namespace subspec
