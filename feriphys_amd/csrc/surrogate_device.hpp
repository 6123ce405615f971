// Device pieces shared by the surrogate's inference and training kernels: the MFMA they use, the
// network's activation and its derivative, the hash that draws training rows.
//
// MFMA used throughout: v_mfma_f32_16x16x32_bf16.  Operand layout (lane l of a wave, s = 0..7):
// A[16 x 32]: row l%16, k = (l/16)*8 + s;  B[32 x 16]: column l%16, k = (l/16)*8 + s;
// C[16 x 16] (4 f32 per lane): rows (l/16)*4 + r, column l%16.
#pragma once

#include "surrogate.hpp"

#pragma clang fp contract(fast)

namespace fp {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The network's activation, a GELU without transcendentals: x s(x) with the normal CDF replaced by
// a C1 piecewise quadratic,
//   s(x) = clamp(0.5 + x (a - b min(|x|, x*)), 0, 1),  a = 1 / x*,  b = 1 / (2 x*^2),
// which reaches 1 (and 0) with zero slope at |x| = x*, so act(x) is exactly x for x >= x* and 0 for
// x <= -x*; x* = 2.46298 minimises max |act(x) - x Phi(x)| (0.0197).  Four VALU operations per
// element (the two clamps ride on a multiply and an FMA): the activation is what the inference
// kernel spends most of its vector instructions on.
constexpr float kXs = 2.4629791631638027f, kA = 0.4060123670374283f, kB = 0.08242302109366773f;
constexpr float kIXs = (float)(1.0 / 2.4629791631638027), kBX = (float)(0.08242302109366773 * 2.4629791631638027);
__device__ __forceinline__ float gelu(float x) {
  const float t = __builtin_amdgcn_fmed3f(fabsf(x) * kIXs, 0.0f, 1.0f);  // min(|x|, x*) / x*
  const float s = __builtin_amdgcn_fmed3f(fmaf(x, fmaf(-kBX, t, kA), 0.5f), 0.0f, 1.0f);
  return x * s;
}
__device__ __forceinline__ float gelu_grad(float x) {
  const float t = __builtin_amdgcn_fmed3f(fabsf(x) * kIXs, 0.0f, 1.0f);
  const float s = __builtin_amdgcn_fmed3f(fmaf(x, fmaf(-kBX, t, kA), 0.5f), 0.0f, 1.0f);
  const float ds = fabsf(x) < kXs ? fmaf(-2.0f * kB, fabsf(x), kA) : 0.0f;  // s'(x) = a - 2 b |x|
  return fmaf(x, ds, s);
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

}  // namespace

}  // namespace fp
