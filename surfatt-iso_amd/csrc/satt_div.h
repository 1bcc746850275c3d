// Correctly rounded quotients and square roots for the sweep kernels.
//
// A quotient n/d: the reciprocal of d refined twice by Newton's step, the
// product with n, one residual correction in fused arithmetic (Markstein's
// scheme), and the hardware's fixup of zeros, infinities and NaN.  This is
// the correctly rounded quotient while |n|, |d| and their quotient stay
// within 2^-500 .. 2^500 (the compiler's own division scales its operands
// first, for the rest of the range); the sweeps' operands are metric
// entries, slownesses and times in radians, kilometres and seconds, their
// largest (time / spacing)^4, about 2^110 at 10^-3 degrees.
// Quotients of one denominator share its reciprocal: 4 instructions each
// beside its 5, where a division of its own takes 11 and, through the carry
// flag of its scaling, cannot be interleaved freely.
// A square root: the reciprocal square root refined by Goldschmidt's
// iteration and two residual corrections, for 2^-900 and more.
// In FP32 the hardware's estimates are within an ulp, so a reciprocal takes
// one Newton step, a quotient the same residual correction and a square root
// one, for magnitudes of 2^-90 .. 2^90, a root's argument to the largest; the
// mixed cell's are at most about (time / spacing)^2, 2^55 at 10^-3 degrees.
// Compared with `/` and sqrtf: no difference for any mantissa of a reciprocal
// or a root, nor, in one run over all of them, for any of the 2^46 pairs of
// mantissas of a quotient.  tests/test_gpu_div.py compares every mantissa of
// the former, 2^24 quotients, and the ends of these ranges.
#pragma once
#include <hip/hip_runtime.h>

namespace satt {

template <typename V>
struct RecipOf {
  V d, r;  // the denominator and its reciprocal, within an ulp
};
using Recip = RecipOf<double>;

__device__ __forceinline__ Recip recip_of(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return {d, r};
}

// n / v.d, correctly rounded.
__device__ __forceinline__ double quot(double n, const Recip &v) {
  const double q = n * v.r;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-v.d, q, n), v.r, q), v.d, n);
}

__device__ __forceinline__ RecipOf<float> recip_of(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return {d, __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r)};
}

__device__ __forceinline__ float quot(float n, const RecipOf<float> &v) {
  const float q = n * v.r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-v.d, q, n), v.r, q), v.d, n);
}

// 1 / d, correctly rounded.
__device__ __forceinline__ double inverse(double d) { return quot(1.0, recip_of(d)); }
__device__ __forceinline__ float inverse(float d) {
  return __builtin_amdgcn_div_fixupf(recip_of(d).r, d, 1.0f);
}

// sqrt(x), correctly rounded; 0 and infinity are their own roots.
__device__ __forceinline__ double root_of(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = y * 0.5;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return x == 0.0 || x == __builtin_inf() ? x : g;
}
__device__ __forceinline__ float root_of(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const float g = x * y;
  const float r = __builtin_fmaf(__builtin_fmaf(-g, g, x), y * 0.5f, g);
  return x == 0.0f || x == __builtin_inff() ? x : r;
}

}  // namespace satt
