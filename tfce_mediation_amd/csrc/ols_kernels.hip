// Permuted mass-univariate OLS t-values on CDNA4 (gfx950).
//
// What is computed (the reference's tval_int, cynumstats.pyx:59-64, applied to
// X[perm] as in vertex_tfce_multiple_regression_randomise.py:105-107):
//   a = (X'X)^-1 X'y,  sigma^2 = |y - X a|^2 / (n - k),
//   se_c = fl32(sqrt(sigma^2 [(X'X)^-1]_cc))  (se is stored as float32, :49),
//   t_c = a_c / se_c.
// How (my design): the design columns split into fixed ones F (the intercept,
// never moved by a permutation) and permuted ones Z.  For a batch of P
// permutations the only large product is Z_p' Y for every p at once - one dense
// contraction [P*rpp x n] . [n x V] on MFMA, rpp = one row per permuted column.
// With L the Cholesky factor of the permuted Gram matrix (X_p'X_p = L L'),
// h = L^-1 X_p'y gives |y - X a|^2 = y'y - |h|^2 and a = L^-T h, so the
// epilogue needs only h_Z = Linv_ZF g_F + Linv_ZZ g_Z per (permutation, element):
//   SSE = r0 - |h_Z|^2 with r0 = y'y - |Linv_FF g_F|^2 precomputed in FP64.
// Y is centred per element first (exact for every coefficient once the model
// holds an intercept; the intercept's own coefficient gets the mean back), so
// the bf16 split loses precision relative to the spread of y, not its offset.
#include "ols_internal.h"
#include "ols_math.h"

namespace tfcehip {

namespace {

__device__ __forceinline__ uint16_t bf16_rne(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// Split x into `pieces` bf16 terms, each the rounding of what is left.
__device__ __forceinline__ void split_bf16(float x, int pieces, uint16_t out[3]) {
  float r = x;
  for (int p = 0; p < 3; ++p) {
    if (p < pieces) {
      out[p] = bf16_rne(r);
      r = r - bf16_f32(out[p]);  // exact
    } else {
      out[p] = 0;
    }
  }
}

// Split a (scaled) value into fp16 hi and lo: hi = fl16(x), lo = fl16(x - hi);
// x - hi is exact in float, so hi + lo carries about 22 significant bits.
__device__ __forceinline__ void split_f16(float x, uint16_t out[3]) {
  const _Float16 hi = (_Float16)x;
  const _Float16 lo = (_Float16)(x - (float)hi);
  out[0] = __builtin_bit_cast(uint16_t, hi);
  out[1] = __builtin_bit_cast(uint16_t, lo);
  out[2] = 0;
}

// Power of two s with max_abs * s in [2^13, 2^14): fp16 operands well inside
// the normal range; exact to undo.
__device__ __forceinline__ float f16_scale(float max_abs) {
  if (!(max_abs > 0.0f) || !(max_abs < INFINITY)) return 1.0f;
  return ldexpf(1.0f, 13 - ilogbf(max_abs));
}

__global__ __launch_bounds__(256) void ols_prep_kernel(OlsPrepArgs a) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= a.Npad) return;
  const bool valid = v < a.V;
  double mu = 0.0;
  if (valid && a.center) {
    for (int i = 0; i < a.n; ++i) mu += (double)a.Y[(int64_t)i * a.ldy + v];
    mu /= (double)a.n;
  }
  float ys = 1.0f;
  if (a.f16) {
    float mx = 0.0f;
    if (valid)
      for (int i = 0; i < a.n; ++i) mx = fmaxf(mx, fabsf((float)((double)a.Y[(int64_t)i * a.ldy + v] - mu)));
    ys = f16_scale(mx);
    if (valid) a.yinv[v] = 1.0f / ys;
  }
  double yy = 0.0;
  const int nkg = a.Kp / 8;
  for (int kg = 0; kg < nkg; ++kg) {
    float vals[8];
    uint16_t pc[3][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = kg * 8 + j;
      float y = 0.0f;
      if (valid && i < a.n) y = (float)((double)a.Y[(int64_t)i * a.ldy + v] - mu);
      vals[j] = y;
      yy += (double)y * (double)y;
      uint16_t s[3];
      if (a.f16)
        split_f16(y * ys, s);
      else
        split_bf16(y, a.pieces, s);
      pc[0][j] = s[0];
      pc[1][j] = s[1];
      pc[2][j] = s[2];
    }
    const int64_t base = ((int64_t)kg * a.Npad + v) * 8;
    float4* dst = reinterpret_cast<float4*>(a.plane32 + base);
    dst[0] = make_float4(vals[0], vals[1], vals[2], vals[3]);
    dst[1] = make_float4(vals[4], vals[5], vals[6], vals[7]);
    for (int p = 0; p < a.pieces; ++p) {
      uint4 w;
      w.x = (uint32_t)pc[p][0] | ((uint32_t)pc[p][1] << 16);
      w.y = (uint32_t)pc[p][2] | ((uint32_t)pc[p][3] << 16);
      w.z = (uint32_t)pc[p][4] | ((uint32_t)pc[p][5] << 16);
      w.w = (uint32_t)pc[p][6] | ((uint32_t)pc[p][7] << 16);
      *reinterpret_cast<uint4*>(a.bf[p] + base) = w;
    }
  }
  if (valid) {
    a.mu[v] = a.center ? mu : 0.0;
    a.yy[v] = yy;
  }
}

__global__ __launch_bounds__(256) void ols_fixed_kernel(OlsFixedArgs a) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= a.V) return;
  double g[kOlsMaxK];
#pragma unroll
  for (int q = 0; q < kOlsMaxK; ++q) g[q] = 0.0;
  for (int i = 0; i < a.n; ++i) {
    const double y = (double)a.plane32[((int64_t)(i >> 3) * a.Npad + v) * 8 + (i & 7)];
#pragma unroll
    for (int q = 0; q < kOlsMaxK; ++q)
      if (q < a.f) g[q] += a.F[i * a.f + q] * y;
  }
  double ss = 0.0;
#pragma unroll
  for (int q = 0; q < kOlsMaxK; ++q) {
    if (q < a.f) {
      double hq = 0.0;
      for (int j = 0; j <= q; ++j) hq += a.LFF[q * a.f + j] * g[j];
      ss += hq * hq;
      a.gF[(int64_t)q * a.V + v] = (float)g[q];
      a.hF[(int64_t)q * a.V + v] = (float)hq;
    }
  }
  a.r0[v] = a.yy[v] - ss;
}

// One workgroup (a wave) per permutation: Gram matrix of X_p = [F, Z[perm]], its
// Cholesky factor and the inverse factor (FP64), stored as float for the
// epilogue, plus [(X'X)^-1]_cc per contrast in FP64.  Bound by latency: the rows
// that the permutation picks are brought to LDS by the whole wave, kFactorRows at
// a time (one lane per sum reading them itself waited for memory twice per row),
// and the factors lie in LDS, a lane per row or column.  Every sum is one chain
// in row order.  250 rows, 4 fixed and 2 permuted columns, 128 permutations: 103 -> 15 us.
constexpr int kFactorRows = 64;

__global__ __launch_bounds__(64) void ols_factor_kernel(OlsFactorArgs a) {
  __shared__ double C[kOlsMaxK * kOlsMaxK];
  __shared__ double sF[kFactorRows][kOlsMaxK], sZ[kFactorRows][kOlsMaxK];
  __shared__ double L[kOlsMaxK][kOlsMaxK], Li[kOlsMaxK][kOlsMaxK];
  const int p = blockIdx.x;
  const int tid = threadIdx.x;
  const int32_t* perm = a.perm ? a.perm + (int64_t)p * a.n : nullptr;
  const int k = a.f + a.m;
  const bool cross = tid < a.f * a.m;
  const int cq = cross ? tid / a.m : 0, cb = cross ? tid % a.m : 0;
  double cs = 0.0;
  for (int i0 = 0; a.f > 0 && a.m > 0 && i0 < a.n; i0 += kFactorRows) {
    const int i = i0 + tid;
    if (i < a.n) {
      const int src = perm ? perm[i] : i;
      const bool ok = src >= 0 && src < a.n;  // NaN from there on if not
      for (int q = 0; q < a.f; ++q) sF[tid][q] = a.F[i * a.f + q];
      for (int b = 0; b < a.m; ++b) sZ[tid][b] = ok ? a.Z[src * a.m + b] : NAN;
    }
    __syncthreads();
    if (cross) {
      const int rows = min(kFactorRows, a.n - i0);
#pragma unroll 8
      for (int r = 0; r < rows; ++r) cs += sF[r][cq] * sZ[r][cb];
    }
    __syncthreads();
  }
  if (cross) C[cq * kOlsMaxK + cb] = cs;
  L[tid / kOlsMaxK][tid % kOlsMaxK] = 0.0;
  Li[tid / kOlsMaxK][tid % kOlsMaxK] = 0.0;
  __syncthreads();
  const auto gram = [&](int i, int j) -> double {
    if (i < a.f && j < a.f) return a.FF[i * a.f + j];
    if (i < a.f) return C[i * kOlsMaxK + (j - a.f)];
    if (j < a.f) return C[j * kOlsMaxK + (i - a.f)];
    return a.ZZ[(i - a.f) * a.m + (j - a.f)];
  };
  const int row = tid < k ? tid : 0;
  double g[kOlsMaxK];
#pragma unroll
  for (int j = 0; j < kOlsMaxK; ++j) g[j] = j < k ? gram(row, j) : 0.0;
#pragma unroll
  for (int j = 0; j < kOlsMaxK; ++j) {
    if (j < k) {
      if (tid == j) {
        double d = g[j];
        for (int q = 0; q < j; ++q) d -= L[j][q] * L[j][q];
        L[j][j] = d > 0.0 ? sqrt(d) : NAN;
      }
      __syncthreads();
      if (tid > j && tid < k) {
        double s = g[j];
        for (int q = 0; q < j; ++q) s -= L[tid][q] * L[j][q];
        L[tid][j] = s / L[j][j];
      }
      __syncthreads();
    }
  }
  if (tid < k) {
    const int j = tid;
    Li[j][j] = 1.0 / L[j][j];
    for (int i = j + 1; i < k; ++i) {
      double s = 0.0;
      for (int q = j; q < i; ++q) s += L[i][q] * Li[q][j];
      Li[i][j] = -s / L[i][i];
    }
  }
  __syncthreads();
  float* out = a.Linv + (int64_t)p * 64;
  out[tid] = (float)Li[tid / kOlsMaxK][tid % kOlsMaxK];
  if (tid < kOlsMaxContrasts) {
    double s = 0.0;
    if (tid < a.n_con)
      for (int j = a.con[tid]; j < k; ++j) s += Li[j][a.con[tid]] * Li[j][a.con[tid]];
    a.dc[(int64_t)p * kOlsMaxContrasts + tid] = s;
  }
  // Block b with columns B: beta = Li' h, and the extra sum of squares of B
  // given the other columns is beta_B' [(X'X)^-1_BB]^-1 beta_B = |C^-1 beta_B|^2
  // with C C' = (X'X)^-1_BB = (Li' Li)_BB; row r of Rb is sum_s C^-1[r][s]
  // Li[.][B_s], so |Rb h|^2 is that sum of squares.
  for (int b = tid; b < a.n_blk && a.Rb; b += 64) {
    int B[kOlsMaxK], w = 0;
    for (int j = 0; j < k; ++j)
      if ((a.blk_mask[b] >> j) & 1u) B[w++] = j;
    double S[kOlsMaxK][kOlsMaxK], C[kOlsMaxK][kOlsMaxK], Ci[kOlsMaxK][kOlsMaxK];
    for (int r = 0; r < w; ++r)
      for (int q = 0; q < w; ++q) {
        double s = 0.0;
        for (int j = (B[r] > B[q] ? B[r] : B[q]); j < k; ++j) s += Li[j][B[r]] * Li[j][B[q]];
        S[r][q] = s;
        C[r][q] = 0.0;
        Ci[r][q] = 0.0;
      }
    for (int j = 0; j < w; ++j) {
      double d = S[j][j];
      for (int q = 0; q < j; ++q) d -= C[j][q] * C[j][q];
      d = d > 0.0 ? sqrt(d) : NAN;
      C[j][j] = d;
      for (int i = j + 1; i < w; ++i) {
        double s = S[i][j];
        for (int q = 0; q < j; ++q) s -= C[i][q] * C[j][q];
        C[i][j] = s / d;
      }
    }
    for (int j = 0; j < w; ++j) {
      Ci[j][j] = 1.0 / C[j][j];
      for (int i = j + 1; i < w; ++i) {
        double s = 0.0;
        for (int q = j; q < i; ++q) s += C[i][q] * Ci[q][j];
        Ci[i][j] = -s / C[i][i];
      }
    }
    float* R = a.Rb + ((int64_t)p * a.n_blk + b) * 64;
    for (int r = 0; r < 8; ++r)
      for (int j = 0; j < 8; ++j) {
        double s = 0.0;
        if (r < w && j < k)
          for (int q = 0; q <= r; ++q) s += Ci[r][q] * Li[j][B[q]];
        R[r * 8 + j] = (float)s;
      }
  }
}

__global__ __launch_bounds__(256) void ols_build_a_kernel(OlsBuildAArgs a) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nkg = a.Kp / 8;
  if (idx >= (int64_t)nkg * a.Mpad) return;
  const int kg = (int)(idx / a.Mpad);
  const int64_t row = idx - (int64_t)kg * a.Mpad;
  const int per_tile = a.tile_rows / a.rpp;
  const int64_t rin = row % a.tile_rows;
  const int p = (int)((row / a.tile_rows) * per_tile + rin / a.rpp), j = (int)(rin % a.rpp);
  const bool used = rin < (int64_t)per_tile * a.rpp;
  float vals[8];
  uint16_t pc[3][8];
#pragma unroll
  for (int jj = 0; jj < 8; ++jj) {
    const int i = kg * 8 + jj;
    float z = 0.0f;
    if (used && p < a.P && j < a.m && i < a.n) {
      const int src = a.perm ? a.perm[(int64_t)p * a.n + i] : i;
      z = (src >= 0 && src < a.n) ? a.Z32[src * a.m + j] : NAN;
    }
    vals[jj] = z;
    uint16_t s[3];
    if (a.f16)
      split_f16(j < 8 ? z * a.zscale[j] : 0.0f, s);
    else
      split_bf16(z, a.pieces, s);
    pc[0][jj] = s[0];
    pc[1][jj] = s[1];
    pc[2][jj] = s[2];
  }
  const int64_t base = ((int64_t)kg * a.Mpad + row) * 8;
  if (a.pieces == 0) {
    float4* dst = reinterpret_cast<float4*>(a.a32 + base);
    dst[0] = make_float4(vals[0], vals[1], vals[2], vals[3]);
    dst[1] = make_float4(vals[4], vals[5], vals[6], vals[7]);
  } else {
    for (int q = 0; q < a.pieces; ++q) {
      uint4 w;
      w.x = (uint32_t)pc[q][0] | ((uint32_t)pc[q][1] << 16);
      w.y = (uint32_t)pc[q][2] | ((uint32_t)pc[q][3] << 16);
      w.z = (uint32_t)pc[q][4] | ((uint32_t)pc[q][5] << 16);
      w.w = (uint32_t)pc[q][6] | ((uint32_t)pc[q][7] << 16);
      *reinterpret_cast<uint4*>(a.abf[q] + base) = w;
    }
  }
}

}  // namespace

hipError_t launch_ols_prep(const OlsPrepArgs& a, hipStream_t s) {
  const int64_t blocks = (a.Npad + 255) / 256;
  hipLaunchKernelGGL(ols_prep_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_ols_fixed(const OlsFixedArgs& a, hipStream_t s) {
  const int64_t blocks = (a.V + 255) / 256;
  hipLaunchKernelGGL(ols_fixed_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_ols_factors(const OlsFactorArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(ols_factor_kernel, dim3(a.P), dim3(64), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_ols_build_a(const OlsBuildAArgs& a, hipStream_t s) {
  const int64_t n = (int64_t)(a.Kp / 8) * a.Mpad;
  hipLaunchKernelGGL(ols_build_a_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace tfcehip

// ---------------------------------------------------------------------------
// FP64 single-design OLS, one thread per element (the reference's numpy path
// for one design: cynumstats.pyx:28-112).  a = invXX_a X'y, residuals, SSE,
// se_j = fl32(sqrt(SSE/(n-k) invXX_se[j][j])), t = a / se.
namespace tfcehip {
namespace {

// Bound by the two reads of Y (the coefficients have to be known before the
// residuals), so nothing but Y may stand in its way: the design's rows come
// through the scalar cache (the same for all lanes; a copy in LDS at the largest
// accepted design is 128 KB and leaves one workgroup per CU), the column count
// is a constant, and the next kDirectRows rows are in flight while the present
// ones are summed.  Every sum is one chain in row order, whatever the launch.
// 2 x 163842 elements, 500 rows, 6 columns: 2720 -> 330 us (4.0 TB/s).
constexpr int kDirectRows = 16;

// f(i, y) for every row, in order.
template <class F>
__device__ __forceinline__ void direct_rows(const float* y, int64_t ld, int n, F f) {
  float cur[kDirectRows], nxt[kDirectRows];
  const int whole = n / kDirectRows * kDirectRows;
  if (whole) {
#pragma unroll
    for (int q = 0; q < kDirectRows; ++q) cur[q] = y[(int64_t)q * ld];
  }
  for (int i = 0; i < whole; i += kDirectRows) {
    if (i + kDirectRows < whole) {
#pragma unroll
      for (int q = 0; q < kDirectRows; ++q) nxt[q] = y[(int64_t)(i + kDirectRows + q) * ld];
    }
#pragma unroll
    for (int q = 0; q < kDirectRows; ++q) f(i + q, (double)cur[q]);
#pragma unroll
    for (int q = 0; q < kDirectRows; ++q) cur[q] = nxt[q];
  }
  for (int i = whole; i < n; ++i) f(i, (double)y[(int64_t)i * ld]);
}

template <int K>
__global__ __launch_bounds__(64) void ols_direct_kernel(OlsDirectArgs a) {
  typedef const __attribute__((address_space(4))) double* Scalars;
  const Scalars X = (Scalars)a.X, Ainv = (Scalars)a.Ainv, Sinv = (Scalars)a.Sinv;
  const int64_t v = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (v >= a.V) return;
  const int n = a.n;
  double xty[K], coef[K];
#pragma unroll
  for (int j = 0; j < K; ++j) xty[j] = 0.0;
  double sy = 0.0, syy = 0.0;
  direct_rows(a.Y + v, a.ldy, n, [&](int i, double y) {
    sy += y;
    syy += y * y;
#pragma unroll
    for (int j = 0; j < K; ++j) xty[j] = fma(X[i * K + j], y, xty[j]);
  });
#pragma unroll
  for (int j = 0; j < K; ++j) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < K; ++q) s = fma(Ainv[j * K + q], xty[q], s);
    coef[j] = s;
  }
  double sse = 0.0;
  direct_rows(a.Y + v, a.ldy, n, [&](int i, double y) {
    double fit = 0.0;
#pragma unroll
    for (int j = 0; j < K; ++j) fit = fma(X[i * K + j], coef[j], fit);
    const double r = y - fit;
    sse = fma(r, r, sse);
    if (a.resid) a.resid[(int64_t)i * a.V + v] = r;
  });
  const double s2 = sse / (double)(n - K);
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const float se = (float)sqrt(s2 * Sinv[j * K + j]);
    if (a.coef) a.coef[(int64_t)j * a.V + v] = coef[j];
    if (a.se) a.se[(int64_t)j * a.V + v] = se;
    if (a.t) a.t[(int64_t)j * a.V + v] = coef[j] / (double)se;
  }
  if (a.sse) a.sse[v] = sse;
  if (a.sumy) a.sumy[v] = sy;
  if (a.sumyy) a.sumyy[v] = syy;
}

// Sobel-type z of the indirect effect from the two path t-values
// (pyfunc.py:150-161, calc_indirect :2678-2709): 0 aroian, 1 sobel, 2 goodman.
__global__ void sobel_kernel(const float* ta, const float* tb, int64_t n, int alg, float ta_const, float* z) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double a = ta ? (double)ta[i] : (double)ta_const;
  z[i] = sobel_z(a, (double)tb[i], alg);
}

}  // namespace

hipError_t launch_ols_direct(const OlsDirectArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.V + 63) / 64));
#define TFCE_DIRECT(K_) case K_: hipLaunchKernelGGL(ols_direct_kernel<K_>, grid, dim3(64), 0, s, a); break
  switch (a.k) {
    TFCE_DIRECT(1);
    TFCE_DIRECT(2);
    TFCE_DIRECT(3);
    TFCE_DIRECT(4);
    TFCE_DIRECT(5);
    TFCE_DIRECT(6);
    TFCE_DIRECT(7);
    TFCE_DIRECT(8);
    default: return hipErrorInvalidValue;
  }
#undef TFCE_DIRECT
  return hipGetLastError();
}

hipError_t launch_sobel(const float* ta, const float* tb, int64_t n, int alg, float ta_const, float* z,
                        hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(sobel_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ta, tb, n, alg, ta_const, z);
  return hipGetLastError();
}

}  // namespace tfcehip

namespace tfcehip {
namespace {
// se[j][v] = fl32(sqrt(sigma2[v] * invXX[j][j]))  (cynumstats.pyx:47-52)
__global__ void se_of_slope_kernel(const double* sigma2, const double* diag, int k, int64_t V, float* se) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V) return;
  for (int j = 0; j < k; ++j) se[(int64_t)j * V + v] = (float)sqrt(sigma2[v] * diag[j]);
}
}  // namespace
// Total sum of squares of calcF (cynumstats.pyx:34): per element, about the
// grand mean of all of Y, in FP64.  Three passes: column sums, the grand mean
// (one workgroup, fixed reduction order), then sum_i (y_iv - mean)^2.
__global__ __launch_bounds__(256) void colsum_kernel(const float* Y, int32_t n, int64_t V, int64_t ldy, double* out) {
  const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (v >= V) return;
  double s = 0.0;
  for (int32_t i = 0; i < n; ++i) s += (double)Y[i * ldy + v];
  out[v] = s;
}

__global__ __launch_bounds__(1024) void grand_mean_kernel(const double* sums, int64_t V, int32_t n, double* mean) {
  __shared__ double red[1024];
  double s = 0.0;
  for (int64_t v = threadIdx.x; v < V; v += 1024) s += sums[v];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) mean[0] = red[0] / ((double)n * (double)V);
}

__global__ __launch_bounds__(256) void tss_kernel(const float* Y, int32_t n, int64_t V, int64_t ldy, const double* mean,
                                                 double* tss) {
  const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (v >= V) return;
  const double m = mean[0];
  double s = 0.0;
  for (int32_t i = 0; i < n; ++i) {
    const double d = (double)Y[i * ldy + v] - m;
    s += d * d;
  }
  tss[v] = s;
}

hipError_t launch_total_ss(const float* Y, int32_t n, int64_t V, int64_t ldy, double* tss, double* mean,
                           hipStream_t s) {
  const unsigned blocks = (unsigned)((V + 255) / 256);
  hipLaunchKernelGGL(colsum_kernel, dim3(blocks), dim3(256), 0, s, Y, n, V, ldy, tss);
  hipLaunchKernelGGL(grand_mean_kernel, dim3(1), dim3(1024), 0, s, tss, V, n, mean);
  hipLaunchKernelGGL(tss_kernel, dim3(blocks), dim3(256), 0, s, Y, n, V, ldy, mean, tss);
  return hipGetLastError();
}

hipError_t launch_se_of_slope(const double* sigma2, const double* diag, int k, int64_t V, float* se,
                              hipStream_t s) {
  if (V <= 0) return hipSuccess;
  hipLaunchKernelGGL(se_of_slope_kernel, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, s, sigma2, diag, k, V, se);
  return hipGetLastError();
}
}  // namespace tfcehip
