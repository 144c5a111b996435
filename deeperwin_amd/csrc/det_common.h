// Pieces shared by the determinant kernels: envelope, orbital rows, in-register LU.
#pragma once
#include "common.h"
#include "kernels.h"
#include <utility>

namespace dwmi {

// Calls f with 0 .. N-1 as compile-time constants (register arrays keep constant indices whatever the body's size).
template <typename F, int... I>
__device__ __forceinline__ void unroll_seq(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unroll_seq(F&& f) {
  unroll_seq(f, std::make_integer_sequence<int, N>{});
}

// Scalar-type generic math (T = float for the FP32/BF16 forms, double for the FP64 form).
__device__ __forceinline__ float dsqrt(float x) { return sqrtf(x); }
__device__ __forceinline__ double dsqrt(double x) { return sqrt(x); }
__device__ __forceinline__ float dtanh(float x) { return tanh_fast(x); }
__device__ __forceinline__ double dtanh(double x) { return tanh(x); }
__device__ __forceinline__ float dexp(float x) { return expf(x); }
__device__ __forceinline__ double dexp(double x) { return exp(x); }

// Spin-major row of electron i's first channel in O (up block, then down block, Cp rows per electron).
__device__ __forceinline__ long orb_row(const Shape& sh, long b, int i) {
  const int dn = sh.n - sh.u;
  return (i < sh.u) ? (b * sh.u + i) * sh.Cp : (long)sh.B * sh.u * sh.Cp + (b * dn + (i - sh.u)) * sh.Cp;
}

// Envelope of electron i of walker b at orbital column col; with GRAD also its gradient in r_i and its
// Laplacian.  Shared by the envelope kernel and the determinant kernels that apply it while reading O.
template <typename T, bool GRAD>
__device__ __forceinline__ void envelope_at(const T* __restrict__ kappa, const T* __restrict__ wenv,
                                            const float* __restrict__ r, const float* __restrict__ R, const Shape& sh,
                                            long b, int i, int col, T& env, T& g0, T& g1, T& g2, T& lenv) {
  const int NO = sh.D * sh.n, s = (i < sh.u) ? 0 : 1;
  const float* ri = r + (b * sh.n + i) * 3;
  const T* kap = kappa + (long)s * sh.I * NO;
  const T* we = wenv + (long)s * sh.I * NO;
  env = T(0);
  g0 = T(0);
  g1 = T(0);
  g2 = T(0);
  lenv = T(0);
#pragma unroll 1
  for (int I = 0; I < sh.I; ++I) {
    const T dx = (T)ri[0] - (T)R[I * 3 + 0], dy = (T)ri[1] - (T)R[I * 3 + 1], dz = (T)ri[2] - (T)R[I * 3 + 2];
    const T rho = dsqrt(dx * dx + dy * dy + dz * dz);
    const T k = kap[I * NO + col];
    const T e = we[I * NO + col] * dexp(-k * rho);
    env += e;
    if constexpr (GRAD) {
      const T coef = -k * e / rho;
      g0 += coef * dx;
      g1 += coef * dy;
      g2 += coef * dz;
      lenv += e * (k * k - T(2) * k / rho);
    }
  }
}

__device__ __forceinline__ double readlane_d(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double wave_max_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ double wave_min_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  return v;
}

// In-register LU of the column-per-lane matrix.  Returns the number of row swaps; perm[] (uniform)
// records the row order; mydiag receives U_jj in lane j.
template <int NMAX>
__device__ __forceinline__ int lu_columns(double (&col)[NMAX], int (&perm)[NMAX], double& mydiag, bool& sing, int n,
                                          int lane) {
  int swaps = 0;
#pragma unroll
  for (int i = 0; i < NMAX; ++i) perm[i] = i;
#pragma unroll
  for (int p = 0; p < NMAX; ++p) {
    if (p < n) {
    double best = -1.0;
    int bidx = p;
#pragma unroll
    for (int i = p; i < NMAX; ++i) {
      if (i < n) {
        const double a = fabs(col[i]);
        if (a > best) {
          best = a;
          bidx = i;
        }
      }
    }
    const int piv = __builtin_amdgcn_readlane(bidx, p);
    const double bval = readlane_d(best, p);
    if (!(bval > 0.0)) sing = true;
    if (piv != p) {
      ++swaps;
#pragma unroll
      for (int i = p + 1; i < NMAX; ++i) {
        if (i == piv) {
          const double t = col[p];
          col[p] = col[i];
          col[i] = t;
          const int tp = perm[p];
          perm[p] = perm[i];
          perm[i] = tp;
        }
      }
    }
    const double pivot = readlane_d(col[p], p);
    if (lane == p) {
      mydiag = col[p];
      const double rp = 1.0 / pivot;  // multipliers by the reciprocal, as LAPACK's dgetf2 scales
#pragma unroll
      for (int i = p + 1; i < NMAX; ++i)
        if (i < n) col[i] = col[i] * rp;
    }
#pragma unroll
    for (int i = p + 1; i < NMAX; ++i) {
      if (i < n) {
        const double li = readlane_d(col[i], p);
        if (lane > p) col[i] -= li * col[p];
      }
    }
    }
  }
  return swaps;
}

template <int NMAX>
__device__ __forceinline__ void finish_slogdet(double mydiag, int swaps, bool sing, int n, int lane, double& logabs,
                                               double& sgn) {
  const bool act = lane < n;
  double lg = act ? log(fabs(mydiag)) : 0.0;
  lg = wave_sum_d(lg);
  const unsigned long long neg = __ballot(act && mydiag < 0.0);
  const int nneg = __popcll(neg) + swaps;
  sgn = (nneg & 1) ? -1.0 : 1.0;
  logabs = lg;
  if (sing) {
    sgn = 0.0;
    logabs = -INFINITY;
  }
}

}  // namespace dwmi
