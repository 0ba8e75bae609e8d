// Device helpers shared by the TFCE kernels.
#pragma once
#include "sqrt_pos.h"
#include "tfce_internal.h"

namespace tfcehip {

// (float)(s^E * HH) for one component: E == 1 is one correctly rounded float
// product (exact in double, as fast_tfce.hpp:77 computes it).  E == 0.5 takes
// the root itself (the hardware's reciprocal root and two residual corrections:
// equal to the library's sqrt for every whole number up to 2^24, checked one by
// one) instead of a random 8 bytes of global memory; any other exponent has
// (double)s^E in the per-adjacency table.
__device__ __forceinline__ float tfce_inc(int size, float HH, float E, const double* sizepow) {
  if (E == 1.0f) return __fmul_rn((float)size, HH);
  if (E == 0.5f) return size > 0 ? __double2float_rn(sqrt_pos((double)size) * (double)HH) : 0.0f;
  return __double2float_rn(sizepow[size] * (double)HH);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// First level l with x > T[l] (T strictly decreasing, L levels), kNever if none.
__device__ __forceinline__ int level_of(float xv, const float* s_T, int L, float T0, float dT) {
  if (!(xv > s_T[L - 1])) return kNever;  // also NaN
  int l = 0;
  if (xv < T0) {
    const float g = (T0 - xv) / dT;  // estimate; fixed up against the table below
    l = g < (float)(L - 1) ? (int)g : L - 1;
    if (l < 0) l = 0;
  }
  while (l > 0 && xv > s_T[l - 1]) --l;
  while (!(xv > s_T[l])) ++l;
  return l;
}

// fl(T^H), correctly rounded (T*T is exact in double).  The reference calls libm
// powf, which is one ulp off for ~0.06% of inputs.
__device__ __forceinline__ float pow_h(float T, float H) {
  if (H == 2.0f) return __fmul_rn(T, T);
  if (H == 1.0f) return T;
  return __double2float_rn(pow((double)T, (double)H));
}

// Fields of a ring-packed row (kSurfRing): six 18-bit indices or positions and
// the 9-bit tail (link byte, row length).
__device__ __forceinline__ void ring_fields(const int4 w, int (&p)[kRingMaxDeg], unsigned& tail) {
  const uint64_t lo = (uint64_t)(uint32_t)w.x | (uint64_t)(uint32_t)w.y << 32;
  const uint64_t hi = (uint64_t)(uint32_t)w.z | (uint64_t)(uint32_t)w.w << 32;
  const uint64_t M = kRingNone;
  p[0] = (int)(lo & M);
  p[1] = (int)((lo >> 18) & M);
  p[2] = (int)((lo >> 36) & M);
  p[3] = (int)(((lo >> 54) | (hi << 10)) & M);
  p[4] = (int)((hi >> 8) & M);
  p[5] = (int)((hi >> 26) & M);
  tail = (unsigned)(hi >> 44) & 0x1ffu;
}

}  // namespace tfcehip
