// Correctly rounded FP64 quotients and square roots for the sweep kernels.
//
// A quotient n/d: the reciprocal of d refined twice by Newton's step, the
// product with n, one residual correction in fused arithmetic (Markstein's
// scheme), and the hardware's fixup of zeros, infinities and NaN.  This is
// the correctly rounded quotient while |n|, |d| and their quotient stay
// within 2^-500 .. 2^500 (the compiler's own division scales its operands
// first, for the rest of the range); the sweeps' operands are metric
// entries, slownesses and times in radians, kilometres and seconds.
// Quotients of one denominator share its reciprocal: 4 instructions each
// beside its 5, where a division of its own takes 11 and, through the carry
// flag of its scaling, cannot be interleaved freely.
// A square root: the reciprocal square root refined by Goldschmidt's
// iteration and two residual corrections, for the same range.
#pragma once
#include <hip/hip_runtime.h>

namespace satt {

struct Recip {
  double d, r;  // the denominator and its reciprocal, within an ulp
};

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

}  // namespace satt
