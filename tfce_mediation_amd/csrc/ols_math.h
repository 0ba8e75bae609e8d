// FP64 square roots of the t and z epilogues.
#pragma once
#include <hip/hip_runtime.h>

#include "sqrt_pos.h"

namespace tfcehip {

// fl32(sqrt(max(x, 0))), NaN for NaN, without a branch: the arguments' ends go
// to the smallest and largest normal doubles, whose roots round to 0 and
// infinity as floats.
__device__ __forceinline__ float sqrt_f32(double x) {
  const float s = (float)sqrt_pos(fmin(fmax(x, 2.2250738585072014e-308), 1.7976931348623157e308));
  return x != x ? (float)x : s;
}

// Sobel-type z of the indirect effect from the two path t-values
// (pyfunc.py:150-161, calc_indirect :2678-2709): 0 aroian, 1 sobel, 2 goodman.
// 1 / sqrt(1/b^2 + 1/a^2 [+ or - 1/(a^2 b^2)]) = sqrt(a^2 b^2 / (a^2 + b^2 [+ or
// - 1])), one root in place of three divisions, a root and a division.  False
// where a t is zero, infinite or NaN (or Goodman's difference not positive):
// sobel_z_general is the formula there, written out as the reference writes it.
__device__ __forceinline__ bool sobel_z_fast(double a, double b, double one, float& z) {
  const double A = a * a, B = b * b;  // exact
  const double N = A * B, nd = N * (A + B + one);
  const double r = __builtin_amdgcn_rsq(nd), h = 0.5 * r;
  double s = nd * r;  // sqrt(N D), z = N / sqrt(N D)
  s = fma(fma(-s, s, nd), h, s);
  double q = fma(fma(-s, r, 1.0), r, r);  // its reciprocal, corrected twice
  q = fma(fma(-s, q, 1.0), q, q);
  z = (float)(N * q);
  return nd > 0.0 && nd < (double)INFINITY;
}

__device__ __forceinline__ double sobel_one(int alg) { return alg == 0 ? 1.0 : (alg == 1 ? 0.0 : -1.0); }

__device__ __forceinline__ float sobel_z_general(double a, double b, int alg) {
  const double ia = 1.0 / (a * a), ib = 1.0 / (b * b), iab = 1.0 / (a * a * b * b);
  double d;
  if (alg == 0) d = ib + ia + iab;
  else if (alg == 1) d = ib + ia;
  else d = ib + ia - iab;
  return (float)(1.0 / sqrt(d));
}

__device__ __forceinline__ float sobel_z(double a, double b, int alg) {
  float z;
  return sobel_z_fast(a, b, sobel_one(alg), z) ? z : sobel_z_general(a, b, alg);
}

}  // namespace tfcehip
