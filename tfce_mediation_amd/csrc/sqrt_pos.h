// FP64 square root by the hardware's reciprocal root.
#pragma once
#include <hip/hip_runtime.h>

namespace tfcehip {

// Square root of a positive, finite double: the hardware's reciprocal square
// root (24 bits and more) and two residual corrections, each squaring its
// error; within 1 ulp of the rounded root (the library's sqrt, with its scaling
// for subnormal arguments, is three times as many instructions).
__device__ __forceinline__ double sqrt_pos(double x) {
  const double r = __builtin_amdgcn_rsq(x), h = 0.5 * r;
  double s = x * r;
  s = fma(fma(-s, s, x), h, s);
  return fma(fma(-s, s, x), h, s);
}

}  // namespace tfcehip
