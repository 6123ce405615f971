// Correctly rounded f32 operations computed without the division instruction sequence.  Those of one
// operand are checked bit for bit against the plain operator on every finite f32 input, on the CPU
// (tests/native) or, where they rest on the gfx950 reciprocal and square root, on the GPU
// (fp_selftest_exact_math); the quotient of two operands as div_by_rcp says.
#pragma once

#ifndef FP_HD
#define FP_HD inline
#endif

namespace fp {

// x / 3.0f, correctly rounded: q0 = x * RN(1/3), then one FMA correction with the exact remainder
// fma(-q0, 3, x).  The zero guard keeps the sign of a zero quotient.
FP_HD float div3_rn(float x) {
  const float third = 0.3333333432674408f;  // RN(1/3) = 0x3eaaaaab
  const float q0 = x * third;
  const float r = __builtin_fmaf(-q0, 3.0f, x);
  return q0 == 0.0f ? q0 : __builtin_fmaf(r, third, q0);
}

// 1.0f / x, correctly rounded.  On gfx950 for |x| in [2^-126, 2^126]: the hardware reciprocal
// (within 1 ulp) refined once by Newton's step with the exact residual fma(-x, r, 1); checked on
// every such input against the division (fp_selftest_exact_math).  Other inputs (zero, subnormal,
// huge, inf, NaN) and host code take the division.
FP_HD float rcp_rn(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  const float ax = __builtin_fabsf(x);
  if (ax >= 0x1p-126f && ax <= 0x1p126f) {
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
  }
#endif
  return 1.0f / x;
}

// sqrt(x), correctly rounded.  On gfx950 for x in [2^-96, FLT_MAX]: the hardware reciprocal square
// root r, g = x r (within 2 ulp) and one Newton step g + (x - g g) r / 2 with the exact residual, one
// transcendental and four other operations (choosing among the hardware square root and its two
// neighbours by their residuals took eight); checked on every such input against the full sequence
// (fp_selftest_exact_math).  Other inputs take the full sequence.
FP_HD float sqrt_in_range(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  const float r = __builtin_amdgcn_rsqf(x), g = x * r;
  return __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * r, g);
#else
  return __builtin_sqrtf(x);
#endif
}
FP_HD float rcp_in_range(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
#else
  return 1.0f / x;
#endif
}
FP_HD float sqrt_rn(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  if (x >= 0x1p-96f && x <= 3.40282347e38f) return sqrt_in_range(x);
#endif
  return __builtin_sqrtf(x);
}

// sqrt(x) and 1 / sqrt(x), each correctly rounded (the reciprocal of the rounded root): one range
// test for both.
FP_HD void sqrt_rcp_rn(float x, float& root, float& inv) {
#ifdef __HIP_DEVICE_COMPILE__
  if (x >= 0x1p-96f && x <= 0x1p96f) {
    root = sqrt_in_range(x);
    inv = rcp_in_range(root);
    return;
  }
#endif
  root = __builtin_sqrtf(x);
  inv = 1.0f / root;
}

// a / b, correctly rounded, given y = RN(1 / b): q = a y and one correction by the exact residual
// a - b q.  The corrected value is within 2^-46 (1 + 2^-24)^2 of a / b, relative, before its one rounding,
// so only pairs whose quotient is that close to a midpoint of two floats could go wrong; the check
// tests/native/div_rcp_check.cpp derives them, all 33,555,480 pairs of significands, and none does.  It
// scales wherever a, b, y, q and the residual (a multiple of ulp(b) ulp(q)) are normal numbers or zero
// with a's sign: callers keep |a| and |b| within [2^-60, 2^60], or say what else holds.  Five operations
// where the compiler's division sequence takes about ten.
FP_HD float div_by_rcp(float a, float b, float y) {
  const float q = a * y;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
FP_HD bool div_range(float x) {
  const float ax = __builtin_fabsf(x);
  return ax >= 0x1p-60f && ax <= 0x1p60f;
}
FP_HD float div_rn(float a, float b) {
#ifdef __HIP_DEVICE_COMPILE__
  if (div_range(a) && div_range(b)) return div_by_rcp(a, b, rcp_in_range(b));
#endif
  return a / b;
}

// x / PI (PI = std::f32::consts::PI = 0x40490fdb), correctly rounded: for x >= 2^-100 the product
// with RN(1/PI) corrected once by the exact remainder fma(-q0, PI, x) (the same method as div3_rn;
// below 2^-104 the remainder is no longer exact), otherwise (tiny, zero, negative, NaN) the
// division itself.
FP_HD float div_pi_in_range(float x) {
  const float pi = 3.14159274101257324f, inv_pi = 0.31830987334251404f;  // 0x40490fdb, RN(1/PI) = 0x3ea2f983
  const float q0 = x * inv_pi;
  return __builtin_fmaf(__builtin_fmaf(-q0, pi, x), inv_pi, q0);
}
FP_HD float div_pi_rn(float x) {
  if (!(x >= 0x1p-100f)) return x / 3.14159274101257324f;
  return div_pi_in_range(x);
}

}  // namespace fp
