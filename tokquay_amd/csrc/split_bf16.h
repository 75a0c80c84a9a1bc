// fp32 operands as three bf16 limbs for the bf16 matrix cores (linear.hip says why and how exact).
#pragma once

#include "tq_internal.h"

namespace tq {
namespace {

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));

// Eight fp32 values as three bf16 limbs: limb l holds the values' l-th bf16 (round to nearest of
// what the limbs before left, an exact subtraction).
__device__ __forceinline__ void split8(const floatx4& lo, const floatx4& hi, uint32x4 (&limb)[3]) {
  float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
  for (int l = 0; l < 3; ++l) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const floatx2 pair = {v[2 * p], v[2 * p + 1]};
      const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, bf16x2));
      limb[l][p] = u;
      if (l < 2) {
        v[2 * p] -= __uint_as_float(u << 16);
        v[2 * p + 1] -= __uint_as_float(u & 0xffff0000u);
      }
    }
  }
}

// The limbs of |v| >= kWhole add up to v; those of a smaller v are off by at most 2^-134, half the smallest bf16
// (the conversion and the MFMA keep bf16 subnormals). An output summed over n products x w is then off by
// at most n 2^-133 max(|x|, |w|).
constexpr float kWhole = 0x1p-110f;

// Whether 0 < |v| < kWhole.
__device__ __forceinline__ bool loses_bits(float v) {
  return 2 * __float_as_uint(v) - 1 < 2 * __builtin_bit_cast(uint32_t, kWhole) - 1;  // 0 wraps to the largest
}

// NaN if any is (v_minimum3_f32, v_maximum3_f32).
__device__ __forceinline__ float min3(float a, float b, float c) {
  return __builtin_elementwise_minimum(__builtin_elementwise_minimum(a, b), c);
}
__device__ __forceinline__ float max3(float a, float b, float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}

// The six limb products that make an fp32 product, smallest first: limb of A, limb of B.
constexpr int kLimbA[6] = {2, 0, 1, 1, 0, 0}, kLimbB[6] = {0, 2, 1, 0, 1, 0};

}  // namespace
}  // namespace tq
