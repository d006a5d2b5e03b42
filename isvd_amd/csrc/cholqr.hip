// CholeskyQR2 for the tall-skinny QR of the pipeline's sketch blocks (and of Z in the TS
// postprocessing): two passes of  W = Y^T Y (MFMA GEMM),  W = R^T R (Cholesky),  Q = Y R^-1
// (MFMA GEMM against the explicit triangular inverse).  One pass leaves an orthogonality error
// of about u kappa(Y)^2; the second pass, on a basis with kappa close to 1, brings it to O(u),
// and the residual ||Y - Q R|| is O(u) ||Y|| as for Householder QR, whenever
// kappa(Y) <~ u^-1/2 (Y. Yamamoto, Y. Nakatsukasa, Y. Yanagisawa, T. Fukaya, "Roundoff error
// analysis of the CholeskyQR2 algorithm", ETNA 44, 2015).  That condition is certified on the
// device: a pivot that is not positive in either factorization, or ||Q1^T Q1 - I||_F > 1/2
// after the first pass, makes the call return false with Y untouched, and the caller runs its
// reference factorization instead.  The l x l steps run in FP64 also for FP32 data.
#include "la.hpp"
#include "mx.hpp"

#include <cstdlib>
#include <type_traits>
#include <vector>

namespace isvd {

namespace {

constexpr int kCqMax = 1024;  // threads at most: n = 128

// 1/d to rounding: the instruction's approximation and two Newton steps
__device__ __forceinline__ double rcp_newton(double d) {
  double w = __builtin_amdgcn_rcp(d);
  w = w * (2.0 - d * w);
  return w * (2.0 - d * w);
}

// One workgroup per l x l block: W (full symmetric storage, upper triangle read) -> R (upper
// Cholesky factor, W = R^T R, lower part zero) and Rinv = R^-1 (upper).  With check, first
// ||W - I||_F is formed and more than 1/2 marks the block failed.  status[b] := 1 on failure
// (non-positive or non-finite pivot); the outputs of a failed block are not used.
//
// The elimination of W = L D L^T and of L X = I in one pass: row i of the working matrix holds
// W's remaining part in columns > k and X = L^-1 in columns <= k, and step k subtracts l_i = W(i,
// k) / d_k times row k from every row i > k (X(i, k) := -l_i).  R = D^(1/2) L^T is row k itself
// over d_k^(1/2), R^-1 = L^-T D^(-1/2) is X^T.  Thread (ti, tj) keeps rows 4 ti .. 4 ti + 3 of
// columns 4 tj .. 4 tj + 3 in registers, so a step is one barrier, the publishing of one row
// through LDS and eight reads of it.  A launch within a decomposition (the matrix in LDS, five
// barriers and a division per column in two passes before): l = 32 40 -> 24 us, 47 65 -> 40, 64 96 ->
// 50, 128 265 -> 146 .. 180 (one block after the FP32 products of the mixed family, at their clock:
// 265).
__global__ __launch_bounds__(kCqMax) void chol_inv_kernel(int n, int n4,
                                                          const double *__restrict__ W,
                                                          double *__restrict__ R,
                                                          double *__restrict__ Rinv, int check,
                                                          int *__restrict__ status) {
  __shared__ __align__(16) double row[2][128];
  __shared__ double dia[128];
  __shared__ double red[kCqMax / 64];
  const int b = blockIdx.x, t = threadIdx.x;
  const double *Wb = W + (i64)b * n * n;
  double *Rb = R + (i64)b * n * n, *Ib = Rinv + (i64)b * n * n;
  const bool live = t < n4 * n4;
  const int ti = live ? t % n4 : 0, tj = live ? t / n4 : 0;
  const int i0 = 4 * ti, j0 = 4 * tj;
  double a[4][4];
  double dev = 0;
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = i0 + p, j = j0 + q;
      double v = i == j ? 1.0 : 0.0;  // rows and columns past n: the identity
      if (i < n && j < n) v = (i <= j) ? Wb[i + (i64)j * n] : Wb[j + (i64)i * n];
      a[p][q] = v;
      const double d = v - (i == j ? 1.0 : 0.0);
      if (live) dev += d * d;
    }
  bool fail = false;
  if (check) {
    for (int off = 32; off > 0; off >>= 1) dev += __shfl_xor(dev, off, 64);
    if ((t & 63) == 0) red[t >> 6] = dev;
    __syncthreads();
    double s = 0;
    for (int w = 0; w < (int)blockDim.x / 64; ++w) s += red[w];
    if (!(s <= 0.25)) fail = true;  // ||W - I||_F > 1/2, or not finite
  }
  for (int kb = 0; kb < n4; ++kb) {
#pragma unroll
    for (int ku = 0; ku < 4; ++ku) {
      const int k = 4 * kb + ku;
      double *v = row[ku & 1];
      if (live && ti == kb) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[j0 + q] = a[ku][q];
      }
      __syncthreads();
      double d = v[k];
      if (!(d > 0.0) || !(d < (double)INFINITY)) {
        fail = true;
        d = 1.0;
      }
      if (t == 0) dia[k] = d;
      const double w = rcp_newton(d);
      double l[4], c[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) l[p] = i0 + p > k ? v[i0 + p] * w : 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = v[j0 + q];
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) a[p][q] -= l[p] * c[q];
      if (tj == kb) {
#pragma unroll
        for (int p = 0; p < 4; ++p) a[p][ku] = i0 + p > k ? -l[p] : a[p][ku];
      }
      // row k of R: the published row over d^(1/2) from the diagonal on
      if (live && ti == kb) {
        const double s = 1.0 / sqrt(d);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (k < n && j0 + q < n) Rb[k + (i64)(j0 + q) * n] = j0 + q >= k ? c[q] * s : 0.0;
      }
    }
  }
  __syncthreads();
  // R^-1(j, i) = X(i, j) / d_i^(1/2) for j <= i, X(i, i) = 1
  if (live) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int i = i0 + p;
      if (i >= n) continue;
      const double s = 1.0 / sqrt(dia[i]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = j0 + q;
        if (j < n) Ib[j + (i64)i * n] = j < i ? a[p][q] * s : (j == i ? s : 0.0);
      }
    }
  }
  if (t == 0) status[b] = fail ? 1 : 0;
}

void chol_inv(i64 n, i64 batch, const double *W, double *R, double *Rinv, int check, int *status) {
  const int n4 = (int)((n + 3) / 4), nt = (n4 * n4 + 63) / 64 * 64;
  hipLaunchKernelGGL(chol_inv_kernel, dim3((unsigned)batch), dim3(nt), 0, ctx().stream, (int)n, n4,
                     W, R, Rinv, check, status);
  LAUNCH_CHECK();
}

}  // namespace

int cholqr_mode() {
  const char *e = std::getenv("ISVD_CHOLQR");
  if (!e) return 0;
  if (e[0] == '0') return 1;
  if (e[0] == '1') return 2;
  return 0;
}

namespace {

// l x l steps in FP64 for either data type: W (T) -> R, R^-1 (FP64), R^-1 also as T for the
// product with the data
template <typename T>
void chol_step(i64 l, i64 batch, const T *w, double *w64, double *r, double *rinv64, T *rinv,
               int check, int *status) {
  const double *wd = w64;
  if constexpr (std::is_same_v<T, double>) {
    wd = w;
  } else {
    convert<double, float>(l, l * batch, w, l, w64, l);
  }
  chol_inv(l, batch, wd, r, rinv64, check, status);
  if constexpr (!std::is_same_v<T, double>) convert<float, double>(l, l * batch, rinv64, l, rinv, l);
}

}  // namespace

template <typename T>
bool cholqr2_rowmajor(i64 m, i64 l, T *Y, i64 ldy, i64 sY, i64 batch, T *R, i64 ldr, i64 sR) {
  ISVD_CHECK(l >= 1 && l <= 128 && m >= l, "CholeskyQR2: needs 1 <= l <= 128 and m >= l");
  constexpr bool dbl = std::is_same_v<T, double>;
  const i64 ll = l * l, ldz = batch * l;
  DBuf<T> w(batch * ll), z(m * ldz), rinv_t(dbl ? 0 : batch * ll);
  DBuf<double> w64(dbl ? 0 : batch * ll), r1(batch * ll), r2(batch * ll), rinv(batch * ll);
  DBuf<int> st(2 * batch);
  T *rinv_data;
  if constexpr (dbl) rinv_data = rinv.get();
  else rinv_data = rinv_t.get();
  // pass 1: W1 = Y^T Y, W1 = R1^T R1, Z^T = R1^-T Y^T
  gram_rows<T>(l, m, Y, ldy, sY, w.get(), batch);
  chol_step<T>(l, batch, w.get(), w64.get(), r1.get(), rinv.get(), rinv_data, 0, st.get());
  apply_upper<T>(l, m, rinv_data, Y, ldy, sY, z.get(), ldz, l, batch);
  // pass 2 on Z, certified by ||Z^T Z - I||_F <= 1/2
  gram_rows<T>(l, m, z.get(), ldz, l, w.get(), batch);
  chol_step<T>(l, batch, w.get(), w64.get(), r2.get(), rinv.get(), rinv_data, 1,
               st.get() + batch);
  std::vector<int> h(2 * batch);
  read_back(h.data(), st.get(), sizeof(int) * 2 * batch);
  for (int v : h)
    if (v) return false;
  apply_upper<T>(l, m, rinv_data, z.get(), ldz, l, Y, ldy, sY, batch);
  // R = R2 R1
  if (R) {
    if constexpr (dbl) {
      gemm<double>('N', 'N', l, l, l, 1.0, r2.get(), l, r1.get(), l, 0.0, R, ldr, batch, ll, ll,
                   sR);
    } else {
      gemm<double>('N', 'N', l, l, l, 1.0, r2.get(), l, r1.get(), l, 0.0, w64.get(), l, batch,
                   ll, ll, ll);
      for (i64 b = 0; b < batch; ++b)
        convert<float, double>(l, l, w64.get() + b * ll, l, R + b * sR, ldr);
    }
  }
  return true;
}

template bool cholqr2_rowmajor<double>(i64, i64, double *, i64, i64, i64, double *, i64, i64);
template bool cholqr2_rowmajor<float>(i64, i64, float *, i64, i64, i64, float *, i64, i64);

}  // namespace isvd
