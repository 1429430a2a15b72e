// Correctly rounded fp32 square root and division in short forms for the value ranges a
// neighbour walk meets.
//
// With -fhip-fp32-correctly-rounded-divide-sqrt the compiler lowers sqrtf and '/' to
// general sequences that handle every input: a square root pre-scales arguments below
// 2^-96 by 2^32 and patches +-0 / +inf afterwards (v_cmp_class); a division range-reduces
// both operands with v_div_scale, post-scales in v_div_fmas and patches special cases in
// v_div_fixup.  Inside the ranges below the following shorter sequences return the same bits
// (checked on the GPU against the compiled general forms: every float for the square root, every
// finite one from 2^-52 on for its reciprocal; for the division every divisor significand against
// 2,047 numerators at the corners of the ranges, and every pair of significands at one pair of
// exponents with selfcheck --exhaustive; rtp_selfcheck_*):
//
//   square root: y = v_rsq_f32(x), s0 = x*y, s = s0 + (x - s0*s0)*(y/2), for x = 0 (y is
//   taken of 2^-96 there), x >= 2^-96 or NaN;
//
//   reciprocal of a divisor d > 0 in [2^-40, 2^40]: y0 = rcp(d), y = y0 + (1 - d*y0)*y0,
//   which is the correctly rounded 1/d for every significand.  The same step from y0 =
//   v_rsq_f32(x), x >= 2^-52, gives the correctly rounded reciprocal of s = sqrtf(x) except where
//   the significand of s is all ones (there the step's tie goes the wrong way);
//
//   division n / d by such a reciprocal: q0 = n*y, q = q0 + (n - d*q0)*y (Markstein, IBM J.
//   Res. Dev. 34(1), 1990: one remainder correction is enough when y is the correctly
//   rounded reciprocal), for d in [2^-40, 2^40] and n = +-0 or |n| in [2^-90, 2^50] with
//   |n|/d in [2^-120, 2^90]: operands and quotient normal, the remainder a multiple of
//   2^(e(n) - 46) >= 2^-136 and so exact even where it is denormal, and exponent differences
//   below the 96 at which v_div_scale starts scaling.
//
// The reciprocal y depends on d alone, so divisions by one divisor share it.
//
// Issue slots of one lane's pair (a quarter-rate v_rsq, v_rcp or v_sqrt counts four): square
// root, reciprocal and three quotients 44 with v_sqrt and its two one-ulp residual tests, a
// v_rcp and two remainder corrections a quotient, 24 in these forms.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rtp {

constexpr uint32_t kSqrtShortMin = 0x0f800000u;  // 2^-96
constexpr uint32_t kDivNumMin = 0x12800000u;     // 2^-90
constexpr float kDivDenMin = 0x1p-40f, kDivDenMax = 0x1p40f;

// Marks a wave-uniform branch taken only when some lane needs a general form: the empty
// volatile statement keeps the compiler from if-converting (always executing) the block.
__device__ __forceinline__ void rare_path()
{
  asm volatile("");
}

// A square root and the raw estimate of its reciprocal.
struct Root {
  float r;  // sqrtf(x) for x = 0, x >= 2^-96 or NaN (NaN for +inf)
  float y;  // v_rsq_f32(x), or of 2^-96 if x is less (root_pair: 0 below 2^-52)
};

__device__ __forceinline__ Root root_short(float x)
{
  // x >= 0 or NaN: the unsigned order of the bits is the order of the values
  const float y = __builtin_amdgcn_rsqf(__uint_as_float(max(__float_as_uint(x), kSqrtShortMin)));
  const float s = x * y, h = 0.5f * y;
  return Root{ __builtin_fmaf(__builtin_fmaf(-s, s, x), h, s), y };
}

// sqrtf(x) for x >= 0: the short form, and the general one for lanes with 0 < x < 2^-96 or
// x = +inf.
__device__ __forceinline__ float sqrt_cr(float x)
{
  float s = root_short(x).r;
  const uint32_t b = __float_as_uint(x);
  const bool general = (b - 1u < kSqrtShortMin - 1u) | (b == 0x7f800000u);
  if (__builtin_amdgcn_ballot_w64(general) != 0) {
    rare_path();
    if (general)
      s = __builtin_sqrtf(x);
  }
  return s;
}

// The root of a pair's squared distance, for quotients by it (root_rcp).  Below 2^-52 (near) root
// and estimate are 0: right for x = 0, where a quotient has to be 0 also when the differences are
// not 0 and their squares underflow, and wrong for the others.
constexpr uint32_t kRootNear = 0x25800000u;  // 2^-52
__device__ __forceinline__ bool root_near(float x) { return __float_as_uint(x) < kRootNear; }
__device__ __forceinline__ Root root_pair(float x)
{
  float y = __builtin_amdgcn_rsqf(x);
  y = root_near(x) ? 0.0f : y;
  const float s = x * y, h = 0.5f * y;
  return Root{ __builtin_fmaf(__builtin_fmaf(-s, s, x), h, s), y };
}

// The reciprocal of a root r = sqrtf(x) from its estimate, for finite x >= 2^-52; wrong in the
// last bit where ones_significand(r).
__device__ __forceinline__ float root_rcp(Root q)
{
  return __builtin_fmaf(__builtin_fmaf(-q.r, q.y, 1.0f), q.y, q.y);
}

__device__ __forceinline__ bool ones_significand(float r)
{
  return (__float_as_uint(r) | 0xff800000u) == 0xffffffffu;
}

// Refined reciprocal of a divisor d in [2^-40, 2^40].
__device__ __forceinline__ float rcp_refined(float d)
{
  const float y0 = __builtin_amdgcn_rcpf(d);
  const float e = __builtin_fmaf(-d, y0, 1.0f);
  return __builtin_fmaf(e, y0, y0);
}

// n / d for d in [2^-40, 2^40] (y = rcp_refined(d)) and n = +-0 or |n| in [2^-90, 2^50]
// with |n|/d in [2^-120, 2^90]; a zero quotient may have either sign (no sum that starts at
// +0 can tell).
__device__ __forceinline__ float div_unsigned_zero(float n, float d, float y)
{
  const float q = n * y;
  return __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
}

// ... with the sign of n, as v_div_fixup gives it.
__device__ __forceinline__ float div_short(float n, float d, float y)
{
  const float q = div_unsigned_zero(n, d, y);
  return __uint_as_float((__float_as_uint(q) & 0x7fffffffu) | (__float_as_uint(n) & 0x80000000u));
}

// (bits << 1) - 2 orders |n| as unsigned with +-0 mapped to the top: the smallest of three
// keys is below kDivNumMin's key exactly when one of the numerators is a nonzero value
// under 2^-90.
__device__ __forceinline__ uint32_t num_key(float n)
{
  return (__float_as_uint(n) << 1) - 2u;
}

__device__ __forceinline__ bool tiny_numerator3(float a, float b, float c)
{
  const uint32_t k = min(min(num_key(a), num_key(b)), num_key(c));
  return k < (kDivNumMin << 1) - 2u;
}

}  // namespace rtp
