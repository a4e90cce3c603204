// The erf GELU and its derivative as the kernels evaluate them (polynomial erf, no library call).
#pragma once

#include <hip/hip_runtime.h>

namespace ccf {

// 1 - erfc(|v| / sqrt2) for h = v / 2.  erfc(sqrt2 |h|) is the eighth power of a polynomial of degree 5 in |h| that is 1 at
// 0, kept within [0, 1]: the eighth root falls so slowly that degree 5 holds where erf itself, as u Q(u^2) on a clamped u,
// took degree 17.  The absolute value and the clamp are modifiers of the instructions.  Exactly 1 beyond |v| of 6.2, and
// for infinities (every partial sum then falls to -inf) and NaN.
// (Coefficients: least maximum of (|v| + 1) times the error over |v| <= 9, by reweighted least squares.)
__device__ __forceinline__ float erf_of_twice(float h) {
  const float a = fabsf(h);
  float q = -6.5160656e-03f;
  q = fmaf(q, a, 3.3375409e-02f);
  q = fmaf(q, a, -9.1669185e-03f);
  q = fmaf(q, a, -1.3857770e-01f);
  q = fmaf(q, a, -1.9951809e-01f);
  q = __builtin_amdgcn_fmed3f(fmaf(q, a, 1.0f), 0.0f, 1.0f);
  const float q2 = q * q, q4 = q2 * q2;
  return fmaf(-q4, q4, 1.0f);
}

// erf-form GELU of v = 2 h: h + |h| erf(|v| / sqrt2).  The caller has h for the price of v: half of a sum is one fused
// multiply-add with half of the other addend.  Measured in fp32 against the exact function over all fp16 values: within
// 3.4e-6 and within 4e-6 |v|.  v * Phi(v) by the polynomial of degree 17 had 5.9e-5 up to |v| of 8, 6.9e-6 |v| beyond its
// clamp and 1.1e-5 |v| at most; the largest error over |v| of either, that one and this, by |v|:
//   to 1e-3 0.9e-7 and 2.4e-7, to 0.01 4e-7 and 1.0e-6, to 0.03 1.2e-6 and 2.3e-6, to 0.1 3.8e-6 and 3.9e-6, to 1 8.4e-6
//   and 3.9e-6, to 2 8.4e-6 and 2.1e-6, to 4 9.5e-6 and 1.3e-6, beyond 1.1e-5 and 2e-7
// So it is the worse one below 0.03, by 2e-4 of the rounding to fp16 that follows, and five times better for pre-activations of
// variance 1 (root mean square 1.2e-6 for 5.9e-6).  NaN for -inf, as the exact form's -inf * 0.  Nine full-rate
// instructions, twelve before; the FFN1 epilogue applies it to 256 values per lane and tile and is bound by this arithmetic.
__device__ __forceinline__ float gelu_erf_of_twice(float h) {
  float g = fmaf(fabsf(h), erf_of_twice(h), h);
  // rounded to fp32 in every kernel: fused with a conversion to fp16 behind it, as the compiler would have it in some of
  // them, the instruction rounds once, and kernels that promise the same bits differ
  asm("" : "+v"(g));
  return g;
}

__device__ __forceinline__ float gelu_erf(float v) { return gelu_erf_of_twice(0.5f * v); }

// Derivative of the erf GELU, Phi(v) + v*phi(v), with the same erf.
__device__ __forceinline__ float gelu_erf_grad(float v) {
  const float half_erf = copysignf(0.5f * erf_of_twice(0.5f * v), v);        // 0.5 * erf(v / sqrt2)
  // phi(v) = exp(-v^2/2) / sqrt(2 pi) = exp2(-v^2 * log2(e)/2) * 0.3989...
  const float pdf = 0.3989422804014327f * __builtin_amdgcn_exp2f(-0.72134752044448170368f * v * v);
  return fmaf(v, pdf, 0.5f + half_erf);
}

}  // namespace ccf
