// mbir_selector.h -- the Bragg selector's arithmetic in the bright-field line update
// (BrightField/BFForwardModel.cpp:851-892): the factor of a rejected entry and the selector
// itself, in fewer instructions than the general root and division, with the same bits.
// tests/test_gpu_selector_math.py compares them with the general forms on the device: the
// root for every mantissa, the quotient for seeded pairs and for the pairs whose quotients lie
// next to the middle of two floats, the selector around its threshold.
#pragma once

#include <hip/hip_runtime.h>

namespace mbir {

// The operands for which root_short and quotient_short round correctly
constexpr float kRejectLo = 0x1p-50f, kRejectHi = 0x1p50f;

// sqrt(a): one Newton step on the hardware reciprocal root, in 5 instructions
__device__ inline float root_short(float a)
{
  const float y = __builtin_amdgcn_rsqf(a);
  const float g = a * y, h = 0.5f * y;
  return __fmaf_rn(__fmaf_rn(-g, g, a), h, g);
}

// n / d: Newton steps on the hardware reciprocal (Markstein 1990), without the scaling and
// special cases of the general form
__device__ inline float quotient_short(float n, float d)
{
  const float r0 = __builtin_amdgcn_rcpf(d);
  const float r = __fmaf_rn(__fmaf_rn(-d, r0, 1.0f), r0, r0);
  const float q0 = n * r;
  const float q1 = __fmaf_rn(__fmaf_rn(-d, q0, n), r, q0);
  return __fmaf_rn(__fmaf_rn(-d, q1, n), r, q1);
}

// dT / (ea sqrt(aw)): 16 instructions instead of 45.  lo and hi take the least and largest
// operand, for the caller to check against kRejectLo and kRejectHi (dT alike).
__device__ inline float rejected_factor(float ea, float aw, float dT, float& lo, float& hi)
{
  const float x = ea * root_short(aw);
  lo = fminf(fminf(lo, aw), x);
  hi = fmaxf(fmaxf(hi, aw), x);
  return quotient_short(dT, x);
}

// The selector |e sqrt(aw)| < T in float
__device__ inline bool kept_by_root(float e, float aw, float T)
{
  return fabsf(e * sqrtf(aw)) < T;
}

// T^2, or not a number where the square may not decide: T not positive, or so small that the
// squares lose bits (one that overflows leaves every entry near)
__device__ inline float square_of(float T) { return T > kRejectLo ? T * T : NAN; }

// The selector by e^2 aw < T2 = square_of(T); near is set where the two lie within 2e-6 of each other
// (or are not numbers) and kept_by_root has to decide.  The squares are off by three
// roundings and |e sqrt(aw)| by two, 4.2e-7 of T2 in all.
__device__ inline bool kept_by_square(float e, float aw, float T2, bool& near)
{
  const float p = (e * aw) * e;
  near |= !(fabsf(p - T2) > 2e-6f * T2);
  return p < T2;
}

}  // namespace mbir
