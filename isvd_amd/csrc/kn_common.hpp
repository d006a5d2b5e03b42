// Pieces shared by the two forms of the Kolmogorov-Nagumo iteration: the l x l chain spread over
// workgroups (smallla.hip) and the whole loop in one launch (kn_loop.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace isvd {

typedef double d4s __attribute__((ext_vector_type(4)));
typedef float f4s __attribute__((ext_vector_type(4)));

template <typename T> struct SM;
template <> struct SM<double> {
  using acc = d4s;
  static __device__ __forceinline__ acc mfma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int g) { return (lane >> 4) + 4 * g; }
};
template <> struct SM<float> {
  using acc = f4s;
  static __device__ __forceinline__ acc mfma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int g) { return 4 * (lane >> 4) + g; }
};

constexpr unsigned kChainSpinLimit = 1u << 22;  // ~4 s of polling
constexpr int kSeriesBlocks = 8;                // Paterson-Stockmeyer blocks of 4 powers
constexpr int kSeriesTerms = 4 * kSeriesBlocks + 1;

// words of a grid barrier's state
enum { kBarCount = 0, kBarAbort = 1 };

// device-coherent load and store (they bypass the per-XCD L2s)
template <typename T>
__device__ __forceinline__ T cld(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void cst(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sum_j c[j] Z^j (j < 4) at entry e, Z^0 = I
template <typename T>
__device__ __forceinline__ T block_at(const T *c, T dl, T z, T z2, T z3) {
  return c[0] * dl + c[1] * z + c[2] * z2 + c[3] * z3;
}

// Paterson-Stockmeyer blocks (of 4 powers) needed for the Taylor series of f and g to reach
// a quarter of the unit roundoff for 4 ||Z||_2 <= rho; 0 when more than kSeriesBlocks would be.
// The tail past degree 4t - 1 is bounded by the tabulated terms up to kSeriesTerms - 1 plus the
// last one again (for rho < 1/2 the terms decay at least geometrically with ratio < 1/2).
template <typename T>
__host__ __device__ inline int series_blocks(const T *coef, double rho) {
  const double eps = (sizeof(T) == 8) ? 0x1p-53 : 0x1p-24;
  if (!(rho < 0.5)) return 0;
  const double x = rho / 4.0;
  double tf[kSeriesTerms], tg[kSeriesTerms];
  double xp = 1.0;
  for (int k = 0; k < kSeriesTerms; ++k) {
    tf[k] = fabs((double)coef[k]) * xp;
    tg[k] = fabs((double)coef[kSeriesTerms + k]) * xp;
    xp *= x;
  }
  // tails from degree k on (suffix sums); the smallest t whose tail from 4t on is small enough
  double rf = tf[kSeriesTerms - 1], rg = tg[kSeriesTerms - 1];
  int best = 0;
  for (int k = kSeriesTerms - 1; k >= 4; --k) {
    rf += tf[k];
    rg += tg[k];
    if ((k & 3) == 0 && k / 4 <= kSeriesBlocks && rf <= 0.25 * eps && rg <= 0.25 * eps)
      best = k / 4;
  }
  return best;
}

// Taylor coefficients of f then g (kSeriesTerms each), rounded to T
template <typename T>
const T *series_table();

}  // namespace isvd
