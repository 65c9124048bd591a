// fp32 quotients without an fp32 division: the arithmetic behind the quantisers' scales and codes (quant_fp8.hip), also compiled for the host.
//
// An IEEE fp32 division is about ten vector instructions.  Markstein's method gives the same bits in three where nothing underflows or overflows on the way:
// a quotient from the rounded reciprocal of the divisor, corrected once by its exact remainder.
#pragma once
#include <hip/hip_runtime.h>

namespace llmmm {

// amax / 448, correctly rounded for amax = 0 and 2^-90 <= amax < infinity.
__host__ __device__ __forceinline__ float scale_of_amax(float amax)
{
  constexpr float y = 1.0f / 448.0f;
  const float     q = amax * y;
  return __builtin_fmaf(__builtin_fmaf(-448.0f, q, amax), y, q);
}

// 1 / s from y, a reciprocal that is at most one ulp off the rounded one (v_rcp_f32): rounded correctly, for 33 pairs of a mantissa of s and a y (of 3 x 2^23)
// to the neighbour.
__host__ __device__ __forceinline__ float refined_reciprocal(float s, float y)
{
  return __builtin_fmaf(__builtin_fmaf(-s, y, 1.0f), y, y);
}

// v / s from y = refined_reciprocal(s, .), with the sign of v: correctly rounded for 2^-69 <= s <= 2^92 where the quotient is at least 2^-11, but for three pairs
// of mantissas (s one of the 33), whose neighbour has the same e4m3 code.  Smaller quotients are off by ulps at most and have the code 0; NaN stays NaN.
__host__ __device__ __forceinline__ float rounded_quotient(float v, float s, float y)
{
  const float q = v * y;
  return __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-s, q, v), y, q), v);
}

}  // namespace llmmm
