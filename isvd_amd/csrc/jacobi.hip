// Small dense SVD / symmetric eigensolver for the l x l problems of the pipeline (l <= 128):
// the Gramian eigendecompositions of orthogonalization / postprocessing (gesvd of a PSD
// matrix), the SVD of the TSQR R factor, and the KN eigendecomposition of Z.
//
// Method: one-sided (Hestenes) Jacobi, parallel round-robin ordering over blocks of two columns.
// One workgroup owns one matrix, held column-major in LDS (128 x 128 FP64 = 128 KiB of the 160
// KiB LDS).  A group of 16 lanes holds the four columns of a block pair in registers through the
// two rounds of cross rotations (and, at the start of a sweep, the one inside the blocks), two
// rotations side by side in each, so that LDS traffic, the workgroup barrier and the wait for both
// are paid every second round.  A sweep with no rotation above the relative threshold ends the
// iteration.  The right factor is not accumulated on the way: the rotations go to a log and
// are replayed on the rows of V by a second kernel, every row in registers of its own lanes.
// A PSD matrix is factored by Cholesky in place first, W = L L^T, and the iteration runs on L,
// whose singular values are the roots of W's: 9-10 sweeps instead of 13-15.
//
// Measured, FP64, 256 x 256 matrices with singular values down to 4 % (one rotation a round, with the
// vectors of V in global memory and every norm summed at every rotation, before): V and U at l = 64
// 618 -> 366 + 47 us, l = 128 4050 -> 1582 + 107 us; PSD at l = 48 485 -> 279 us, l = 128 3084 -> 1683
// us.  Bound by instruction issue: the vector unit is busy 50 % (l = 64, one wave per SIMD) to 60 %
// (l = 128, two) of the time, the rest waits for LDS, barriers and dependent FP64 results; four groups
// of lanes per pair instead of two, or eight lanes a group, were slower.
#include "la.hpp"

#include <algorithm>
#include <type_traits>

#include "dpp.hpp"

#include <cfloat>

namespace isvd {

namespace {

template <typename T> struct Eps;
template <> struct Eps<double> {
  static constexpr double v = DBL_EPSILON, least = DBL_MIN;
  static constexpr int exponent = 0;  // see the load
};
template <> struct Eps<float> {
  static constexpr float v = FLT_EPSILON, least = FLT_MIN;
  static constexpr int exponent = 22;
};

constexpr int kMaxSweeps = 40;
// Sweeps the rotation log holds.  Ten or eleven are the rule; columns that collapse onto each other can
// take more, and the rotations so far are then replayed on V before the log starts over.
constexpr int kLogSweeps = 16;
// Bytes the logs of one launch may take: a round of the CUs at n = 128 (256 problems of 2.1 MB in
// FP64), several below.  Larger batches go in several launches.
constexpr size_t kLogBytes = 640ull << 20;
// 16 lanes per block pair, each holding every 16th row of its four columns
constexpr int kTpp = 16;
constexpr int kMaxThreads = 512;  // n = 128: 32 groups

// x^(-1/2): FP64 the hardware's approximation (better than 2^-23) through one step of third order, FP32
// the hardware's (1 ulp)
__device__ __forceinline__ double rsq(double x) {
  const double r = __builtin_amdgcn_rsq(x), e = 1.0 - (x * r) * r;
  return r + (r * e) * (0.375 * e + 0.5);
}
__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }

// rows per lane for an n x n problem (a power of two)
inline int jacobi_rpl(i64 n) {
  int r = 1;
  while (r * kTpp < n) r *= 2;
  return r;
}
// groups (block pairs) of an n-column problem: blocks of two columns, an even number of them
__host__ __device__ inline int jacobi_groups(int n) { return (n + 3) / 4; }

// round-robin (circle method) pairing of np players (np even), round r in [0, np-1), table
// k in [0, np/2): player m = np - 1 stays at table 0, the others turn (r, k < m: no modulo)
__device__ __forceinline__ void rr_pair(int np, int r, int k, int &p, int &q) {
  const int m = np - 1;
  if (k == 0) {
    p = r;
    q = m;
  } else {
    p = (r + k >= m) ? r + k - m : r + k;
    q = (r >= k) ? r - k : r - k + m;
  }
}

// The rotation log of one problem, 2 g slots a sweep (g groups) of four times g rotations: in slot
// 0, for group k, the two rotations inside the blocks it starts with, (p0, p1), (q0, q1); in slot
// 1 + r, r < 2 g - 1, the four cross rotations of its block pair in outer round r, (p0, q0),
// (p1, q1), (p0, q1), (p1, q0).
// A rotation: cos and sin in FP64.  In FP32 t = tan(theta / 2) stands for the cosine, c = 1 - s t: next
// to 1 it has the digits that a cosine rounds away, a few hundred rotations of which had moved the
// singular values by up to n units of roundoff.
template <typename T>
struct Rot {
  T c, s;
  static __device__ Rot none() { return {T(sizeof(T) == 8 ? 1 : 0), T(0)}; }
  __device__ __forceinline__ void turn(T &a, T &b) const {
    const T x = a, y = b;
    if constexpr (sizeof(T) == 8) {
      a = c * x - s * y;
      b = s * x + c * y;
    } else {
      a = x - s * (c * x + y);
      b = y + s * (x - c * y);
    }
  }
};
__host__ __device__ inline i64 log_entries(int groups) {
  return (i64)kLogSweeps * 2 * groups * groups * 4;
}

// One row of V through `slots` slots of the rotation log lg: row i of V is e_i^T (resume: row i of V as
// it is) through the rotations in order.  A row lives in the registers of consecutive lanes (groups of
// them, padded to a power of two), lane k holding the entries of the block pair at table k, and
// between outer rounds the blocks move to the next table as the players of the circle do: p to the
// left, q to the right, turning at both ends.  No barrier, no LDS; the log is read AHEAD outer rounds
// ahead.  Column j of the row is stored as column rank[j] (rank null: j).
template <typename T>
__device__ __forceinline__ T from_next(T v) { return dpp_mov<0x130>(v); }  // lane i: lane i + 1's
template <typename T>
__device__ __forceinline__ T from_prev(T v) { return dpp_mov<0x138>(v); }  // lane i: lane i - 1's

template <typename T, int AHEAD>
__device__ __forceinline__ void replay_row(int n, int k, int row, const Rot<T> *lg, int slots,
                                           bool resume, const int *rank, T *V, i64 ldv) {
  const int groups = jacobi_groups(n), blocks = 2 * groups;
  const bool live = k < groups;
  const int kc = live ? k : 0;
  // the entries of this lane's blocks in round 0: P = k, Q = last block (k = 0) or blocks - 1 - k
  const int P = kc, Q = kc == 0 ? blocks - 1 : blocks - 1 - kc;
  auto entry = [&](int col) -> T {
    if (!resume) return T(row == col);
    return row < n && col < n ? V[row + (i64)col * ldv] : T(0);
  };
  T p0 = entry(2 * P), p1 = entry(2 * P + 1), q0 = entry(2 * Q), q1 = entry(2 * Q + 1);
  struct Slot {
    Rot<T> r[4];
  };
  auto fetch = [&](int i) {
    const int c = i < slots ? i : slots - 1;
    Slot v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v.r[j] = lg[((i64)c * 4 + j) * groups + kc];
    return v;
  };
  if (slots > 0) {
    Slot buf[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) buf[a] = fetch(a);
    int slot = 0;  // of the sweep
    for (int i0 = 0; i0 < slots; i0 += AHEAD) {
#pragma unroll
      for (int a = 0; a < AHEAD; ++a) {
        const Slot s = buf[a];
        buf[a] = fetch(i0 + a + AHEAD);
        if (i0 + a < slots) {
          if (slot == 0) {
            s.r[0].turn(p0, p1);
            s.r[1].turn(q0, q1);
          } else {
            s.r[0].turn(p0, q0);
            s.r[1].turn(p1, q1);
            s.r[2].turn(p0, q1);
            s.r[3].turn(p1, q0);
            if (groups > 1) {
              // p_k := p_{k+1}, p_last := q_last; q_k := q_{k-1} (k >= 2), q_1 := p_0; q_0 stays
              const T np0 = from_next(p0), np1 = from_next(p1);
              const T nq0 = from_prev(k == 0 ? p0 : q0), nq1 = from_prev(k == 0 ? p1 : q1);
              const bool last = k == groups - 1;
              const T lp0 = last ? q0 : np0, lp1 = last ? q1 : np1;
              q0 = k == 0 ? q0 : nq0;
              q1 = k == 0 ? q1 : nq1;
              p0 = lp0;
              p1 = lp1;
            }
          }
          slot = slot + 1 == blocks ? 0 : slot + 1;
        }
      }
    }
  }
  if (row >= n || !live) return;
  // whole sweeps leave every block where it started
  auto store = [&](int col, T v) {
    if (col < n) V[row + (i64)(rank ? rank[col] : col) * ldv] = v;
  };
  store(2 * P, p0);
  store(2 * P + 1, p1);
  store(2 * Q, q0);
  store(2 * Q + 1, q1);
}

// lanes a row takes
__host__ __device__ inline int replay_lanes(int groups) {
  int seg = 1;
  while (seg < groups) seg *= 2;
  return seg;
}

enum { kGeneral = 0, kSymmetric = 1, kPsd = 2 };
// per problem: the columns' ranks, the sweeps in the log, whether V holds those before it
constexpr int kOrder = 132, kOrderSweeps = 128, kOrderResume = 129;

// kGeneral: SVD of A (general n x n).  kSymmetric: symmetric eigendecomposition of the matrix whose
// upper triangle is stored in A, computed as the SVD of sym(A) + c I with c = 2 ||sym(A)||_F.
// kPsd: SVD of a symmetric positive semi-definite A (upper triangle), by the SVD of its Cholesky
// factor where every pivot stays above rounding, else of A itself.
// The columns are padded with zero rows to 16 RPL and with zero columns to 4 groups (rotations
// keep both zero), so the round loop has no bounds.  blockDim.x = 16 lanes per group, rounded up
// to whole waves.
template <typename T, int RPL>
__global__ __launch_bounds__(kMaxThreads) void svd_jacobi_kernel(
    int n, int mode, const T *__restrict__ A, i64 lda, i64 sA, T *__restrict__ sig, i64 lds,
    T *__restrict__ U, i64 ldu, i64 sU, T *V, i64 ldv, i64 sV, Rot<T> *__restrict__ log,
    int *__restrict__ order, T *__restrict__ shift_out) {
  extern __shared__ unsigned char smem_raw[];
  // leading dimension 16 RPL + 1: the columns a wave works on start in different banks
  T *G = reinterpret_cast<T *>(smem_raw);
  __shared__ T red[kMaxThreads / 64];
  __shared__ T nrm[128];  // squared column norms during the sweeps, then the norms
  __shared__ int rank_of[128];
  __shared__ int n_rot;
  __shared__ T shift_sh;
  __shared__ int exp_sh;

  const int b = blockIdx.x;
  const int tid = threadIdx.x;
  const int nt = blockDim.x, waves = nt / 64;
  const T *Ab = A + (i64)b * sA;
  const int groups = jacobi_groups(n), cols = 4 * groups, blocks = 2 * groups;
  const int grp = tid / kTpp, sub = tid % kTpp;
  const bool live = grp < groups;
  constexpr int R = kTpp * RPL;  // padded rows
  constexpr int ld = R + 1;

  // ---- load (rows n .. R-1 and columns n .. zero) ----
  auto load = [&](bool upper, int sh) {
    for (int e = tid; e < R * cols; e += nt) {
      const int i = e % R, j = e / R;
      T v = T(0);
      if (i < n && j < n)
        v = (upper && i > j) ? Ab[j + (i64)i * lda] : Ab[i + (i64)j * lda];
      G[i + j * ld] = ldexp(v, -sh);
    }
    __syncthreads();
  };
  load(mode != kGeneral, 0);
  // The largest entry to 2^(exponent - 1) .. 2^exponent, by a power of two (exactly): the squares of
  // squared norms stay below overflow, and above underflow for columns down to 1e-77 (FP32: 1e-16)
  // of the largest.  Everything below is on the scaled matrix up to what is stored.
  {
    T top = 0;
    for (int e = tid; e < R * cols; e += nt) top = fmax(top, fabs(G[e % R + (e / R) * ld]));
    for (int off = 32; off; off >>= 1) top = fmax(top, __shfl_xor(top, off, 64));
    if ((tid & 63) == 0) red[tid >> 6] = top;
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < waves; ++w) top = fmax(top, red[w]);
      int ex = Eps<T>::exponent;
      if (top > T(0) && top < T(INFINITY)) (void)frexp(top, &ex);
      exp_sh = ex - Eps<T>::exponent;
    }
    __syncthreads();
  }
  const int sh = exp_sh;
  for (int e = tid; e < R * cols; e += nt) {
    T &g = G[e % R + (e / R) * ld];
    g = ldexp(g, -sh);
  }
  __syncthreads();
  if (mode == kSymmetric) {
    // c = 2 ||A||_F (+1 when A == 0), deterministic block reduction
    T part = 0;
    for (int e = tid; e < n * n; e += nt) {
      const T g = G[e % n + (e / n) * ld];
      part += g * g;
    }
    part = lane_group_sum(part, 64);
    if ((tid & 63) == 0) red[tid >> 6] = part;
    __syncthreads();
    if (tid == 0) {
      T s = 0;
      for (int w = 0; w < waves; ++w) s += red[w];
      T c = T(2) * sqrt(s);
      if (c == T(0)) c = T(1);
      shift_sh = c;
    }
    __syncthreads();
    for (int i = tid; i < n; i += nt) G[i + i * ld] += shift_sh;
    __syncthreads();
  }
  bool factored = false;
  if (mode == kPsd) {
    // L D L^T in place, right-looking on the lower triangle, one barrier a step (column k stays
    // unscaled until the end); a pivot not above n u A(k, k) is rounding, and A is taken itself
    for (int j = tid; j < n; j += nt) nrm[j] = Eps<T>::v * T(n) * G[j + j * ld];
    __syncthreads();
    factored = true;
    const int i = tid % R, jg = tid / R, js = nt / R;
    for (int k = 0; k < n; ++k) {
      const T d = G[k + k * ld];
      if (!(d > nrm[k]) || !(d < T(INFINITY))) {
        factored = false;
        break;
      }
      const T w = T(1) / d;
      if (jg < js && i > k && i < n) {
        const T lik = G[i + k * ld] * w;
        for (int j = k + 1 + jg; j <= i; j += js) G[i + j * ld] -= lik * G[j + k * ld];
      }
      __syncthreads();
    }
    if (factored) {
      for (int e = tid; e < R * n; e += nt) {
        const int r = e % R, j = e / R;
        if (r != j) G[r + j * ld] = r > j ? G[r + j * ld] / sqrt(G[j + j * ld]) : T(0);
      }
      __syncthreads();
      for (int j = tid; j < n; j += nt) G[j + j * ld] = sqrt(G[j + j * ld]);
      __syncthreads();
    } else {
      __syncthreads();
      load(true, sh);
    }
  }

  // Rotations down to n / 4 units of roundoff in FP64, 4 units (the dot products are good to about one)
  // in FP32 and below n = 16: vectors are off by as much over the gap of their singular values.  FP64,
  // PSD with 64 and 128 columns, whole postprocessing and distance of the vectors: n units 476 us, 1000
  // and 1830 us, 5900; n / 2 480, 645 and 1825, 3060; n / 4 481, 460 and 1830, 1850; 4 units 490, 372
  // and 1905, 1160.  (One column pair at a time with n units, on W itself: 750 and 4080.)
  const T tol = (sizeof(T) == 4 || n < 16 ? T(4) : T(0.25) * T(n)) * Eps<T>::v;
  const T tol2 = tol * tol;
  // Two rotations side by side, columns (a0, b0) and (a1, b1) with squared norms na, nb.  With
  // d = nb - na and h = 2 gamma, d : h = cot(2 theta): r = (d^2 + h^2)^(-1/2), c^2 = (1 + |d| r) / 2,
  // s = sign(d) h r / (2 c).  A pair with d^2 + h^2 below the smallest normal number is not rotated
  // (both columns are as good as zero).  (With divisions and the library's roots: 110 ns more a round.)
  typedef T Col[RPL];
  int rotated = 0;
  auto sum_sq = [&](const Col &x) {
    T v = 0;
#pragma unroll
    for (int u = 0; u < RPL; ++u) v += x[u] * x[u];
    return lane_group_sum(v, kTpp);
  };
  auto rot2 = [&](Col &a0, Col &b0, T &na0, T &nb0, Col &a1, Col &b1, T &na1, T &nb1,
                  Rot<T> *out) {
    T g0 = 0, g1 = 0;
#pragma unroll
    for (int u = 0; u < RPL; ++u) {
      g0 += a0[u] * b0[u];
      g1 += a1[u] * b1[u];
    }
    g0 = lane_group_sum(g0, kTpp);
    g1 = lane_group_sum(g1, kTpp);
    const T d0 = nb0 - na0, h0 = T(2) * g0, q0 = d0 * d0 + h0 * h0;
    const T d1 = nb1 - na1, h1 = T(2) * g1, q1 = d1 * d1 + h1 * h1;
    // |gamma| > tol sqrt(alpha beta), compared in squares
    const bool n0 = g0 * g0 > tol2 * (na0 * nb0) && q0 >= Eps<T>::least;
    const bool n1 = g1 * g1 > tol2 * (na1 * nb1) && q1 >= Eps<T>::least;
    Rot<T> r0 = Rot<T>::none(), r1 = r0;
    if (n0 || n1) {
      auto angle = [&](bool need, T d, T h, T q, T &na, T &nb) {
        const T r = rsq(q), c2 = T(0.5) + T(0.5) * fabs(d) * r, z = rsq(c2);
        const T c = need ? c2 * z : T(1), sa = T(0.5) * h * r * z;
        const T s = need ? (d >= T(0) ? sa : -sa) : T(0);
        const T g2 = c * s * h, cc = c * c, ss = s * s;
        const T xa = (cc * na - g2) + ss * nb, xb = (ss * na + g2) + cc * nb;
        na = fmax(xa, T(0));
        nb = fmax(xb, T(0));
        if constexpr (sizeof(T) == 8) return Rot<T>{c, s};
        else return Rot<T>{s * __builtin_amdgcn_rcpf(T(1) + c), s};
      };
      r0 = angle(n0, d0, h0, q0, na0, nb0);
      r1 = angle(n1, d1, h1, q1, na1, nb1);
#pragma unroll
      for (int u = 0; u < RPL; ++u) {
        r0.turn(a0[u], b0[u]);
        r1.turn(a1[u], b1[u]);
      }
      rotated = 1;
    }
    if (log && sub == 0 && live) {
      out[0] = r0;
      out[groups] = r1;
    }
  };
  Rot<T> *lg = log ? log + (i64)b * log_entries(groups) : nullptr;
  int logged = 0;  // sweeps in the log
  bool resume = false;
  for (int sweep = 0; sweep < kMaxSweeps; ++sweep) {
    if (log && logged == kLogSweeps) {
      const int lane = tid & 63, seg = replay_lanes(groups), rows = 64 / seg;
      for (int r0 = (tid >> 6) * rows; r0 < n; r0 += waves * rows)
        replay_row<T, 2>(n, lane % seg, r0 + lane / seg, lg, logged * blocks, resume, nullptr,
                         V + (i64)b * sV, ldv);
      resume = true;
      logged = 0;
      __syncthreads();
    }
    if (tid == 0) n_rot = 0;
    rotated = 0;
    for (int r = 0; r < blocks - 1; ++r) {
      int P = 0, Q = 1;
      if (live) rr_pair(blocks, r, grp, P, Q);
      Rot<T> *out = lg + ((i64)logged * blocks + 1 + r) * 4 * groups + grp;
      if (live) {
        T *cp = G + 2 * P * ld + sub, *cq = G + 2 * Q * ld + sub;
        Col p0, p1, q0, q1;
#pragma unroll
        for (int u = 0; u < RPL; ++u) {
          p0[u] = cp[u * kTpp];
          p1[u] = cp[ld + u * kTpp];
          q0[u] = cq[u * kTpp];
          q1[u] = cq[ld + u * kTpp];
        }
        T np0, np1, nq0, nq1;
        if (r == 0) {
          // squared norms afresh; within the sweep each rotation updates its two (a sweep without a
          // rotation, which ends the iteration, thus tested every pair against norms of its
          // columns; the norm of a column that collapses onto another is rounding until then, and
          // a rotation with it no more than a needless one); the rotations inside the blocks
          np0 = sum_sq(p0);
          np1 = sum_sq(p1);
          nq0 = sum_sq(q0);
          nq1 = sum_sq(q1);
          rot2(p0, p1, np0, np1, q0, q1, nq0, nq1, lg + (i64)logged * blocks * 4 * groups + grp);
        } else {
          np0 = nrm[2 * P];
          np1 = nrm[2 * P + 1];
          nq0 = nrm[2 * Q];
          nq1 = nrm[2 * Q + 1];
        }
        rot2(p0, q0, np0, nq0, p1, q1, np1, nq1, out);
        rot2(p0, q1, np0, nq1, p1, q0, np1, nq0, out + 2 * groups);
#pragma unroll
        for (int u = 0; u < RPL; ++u) {
          cp[u * kTpp] = p0[u];
          cp[ld + u * kTpp] = p1[u];
          cq[u * kTpp] = q0[u];
          cq[ld + u * kTpp] = q1[u];
        }
        // (every lane of the group writes the same four values)
        nrm[2 * P] = np0;
        nrm[2 * P + 1] = np1;
        nrm[2 * Q] = nq0;
        nrm[2 * Q + 1] = nq1;
      }
      __syncthreads();
    }
    if (rotated && sub == 0) n_rot = 1;
    __syncthreads();
    const int go = n_rot;
    __syncthreads();
    if (go == 0) break;
    ++logged;
  }

  // ---- singular values (column norms), ranks for descending order ----
  for (int j = tid / 64; j < n; j += waves) {
    T a = 0;
    for (int i = tid % 64; i < n; i += 64) a += G[i + j * ld] * G[i + j * ld];
    a = lane_group_sum(a, 64);
    if ((tid & 63) == 0) nrm[j] = sqrt(a);
  }
  __syncthreads();
  for (int j = tid; j < n; j += nt) {
    int rk = 0;
    const T sj = nrm[j];
    for (int i = 0; i < n; ++i) {
      const T si = nrm[i];
      rk += (si > sj) || (si == sj && i < j);
    }
    rank_of[j] = rk;
  }
  __syncthreads();
  for (int j = tid; j < n; j += nt)
    sig[(i64)b * lds + rank_of[j]] = ldexp(factored ? nrm[j] * nrm[j] : nrm[j], sh);
  if (mode == kSymmetric && tid == 0 && shift_out) shift_out[b] = ldexp(shift_sh, sh);
  if (U) {
    T *Ub = U + (i64)b * sU;
    for (int e = tid; e < n * n; e += nt) {
      const int i = e % n, j = e / n;
      const T sj = nrm[j];
      Ub[i + (i64)rank_of[j] * ldu] = (sj > T(0)) ? G[i + j * ld] / sj : T(0);
    }
  }
  if (order) {
    for (int j = tid; j < n; j += nt) order[b * kOrder + j] = rank_of[j];
    if (tid == 0) {
      order[b * kOrder + kOrderSweeps] = logged;
      order[b * kOrder + kOrderResume] = resume;
    }
  }
}

// V of the SVD from the rotation log, a row per `seg` lanes, the log read eight outer rounds ahead.
// 128 x 128 FP64, 10 sweeps: 107 us (64 x 64: 47 us).
template <typename T>
__global__ __launch_bounds__(256) void jacobi_replay_kernel(int n, int seg,
                                                            const Rot<T> *__restrict__ log,
                                                            const int *__restrict__ order, T *V,
                                                            i64 ldv, i64 sV) {
  const int groups = jacobi_groups(n);
  const int b = blockIdx.y, lane = threadIdx.x & 63;
  const int row = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 / seg) + lane / seg;
  const int *o = order + b * kOrder;
  replay_row<T, 8>(n, lane % seg, row, log + (i64)b * log_entries(groups),
                   o[kOrderSweeps] * 2 * groups, o[kOrderResume] != 0, o, V + (i64)b * sV, ldv);
}

// eigenvalues ascending from the shifted SVD: w[j] = sig[n-1-j] - c, Z[:, j] = U[:, n-1-j]
template <typename T>
__global__ void syev_finish_kernel(int n, const T *sig, const T *shift, const T *Usrt, T *w, T *Z,
                                   i64 ldz) {
  const T c = shift[0];
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n * n; e += gridDim.x * blockDim.x) {
    const int i = e % n, j = e / n;
    Z[i + (i64)j * ldz] = Usrt[i + (i64)(n - 1 - j) * n];
    if (i == 0) w[j] = sig[n - 1 - j] - c;
  }
}

template <typename T, int RPL>
void launch_rpl(i64 n, int mode, const T *A, i64 lda, i64 sA, T *s, i64 lds, T *U, i64 ldu, i64 sU,
                T *V, i64 ldv, i64 sV, i64 batch, Rot<T> *log, int *order, T *shift_out) {
  const int groups = jacobi_groups((int)n);
  const size_t shmem = sizeof(T) * (size_t)(kTpp * RPL + 1) * (size_t)(4 * groups);
  const int nt = (groups * kTpp + 63) / 64 * 64;
  auto kern = svd_jacobi_kernel<T, RPL>;
  HIP_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)shmem));
  hipLaunchKernelGGL(kern, dim3((unsigned)batch), dim3(nt), shmem, ctx().stream, (int)n, mode, A,
                     lda, sA, s, lds, U, ldu, sU, V, ldv, sV, log, order, shift_out);
  LAUNCH_CHECK();
}

template <typename T>
void launch_svd(i64 n, int mode, const T *A, i64 lda, i64 sA, T *s, i64 lds, T *U, i64 ldu,
                i64 sU, T *V, i64 ldv, i64 sV, i64 batch, T *shift_out) {
  ISVD_CHECK(n >= 1 && n <= 128, "small SVD supports 1 <= n <= 128 (got %lld)", n);
  const int groups = jacobi_groups((int)n), seg = replay_lanes(groups);
  i64 chunk = batch;
  if (V) {
    const i64 most = (i64)(kLogBytes / (sizeof(Rot<T>) * (size_t)log_entries(groups)));
    chunk = std::min(chunk, std::min(most, (i64)65535));
  }
  // the logs and, behind them, the orders: one allocation (each and its release take the host about 5 us)
  const i64 entries = V ? chunk * log_entries(groups) : 0;
  DBuf<Rot<T>> buf(V ? entries + ceil_div(chunk * kOrder * (i64)sizeof(int), sizeof(Rot<T>)) : 0);
  Rot<T> *log = buf.get();
  int *order = V ? reinterpret_cast<int *>(log + entries) : nullptr;
  for (i64 b0 = 0; b0 < batch; b0 += chunk) {
    const i64 nb = std::min(chunk, batch - b0);
    T *Vb = V ? V + b0 * sV : nullptr, *Ub = U ? U + b0 * sU : nullptr;
#define ISVD_JAC(R)                                                                             \
  launch_rpl<T, R>(n, mode, A + b0 * sA, lda, sA, s + b0 * lds, lds, Ub, ldu, sU, Vb, ldv, sV, nb, \
                   log, order, shift_out)
    switch (jacobi_rpl(n)) {
      case 1: ISVD_JAC(1); break;
      case 2: ISVD_JAC(2); break;
      case 4: ISVD_JAC(4); break;
      default: ISVD_JAC(8); break;
    }
#undef ISVD_JAC
    if (!V) continue;
    const int rows = 4 * (64 / seg);  // per workgroup
    hipLaunchKernelGGL(jacobi_replay_kernel<T>,
                       dim3((unsigned)((n + rows - 1) / rows), (unsigned)nb), dim3(256), 0,
                       ctx().stream, (int)n, seg, (const Rot<T> *)log,
                       (const int *)order, Vb, ldv, sV);
    LAUNCH_CHECK();
  }
}

}  // namespace

template <typename T>
void svd_small(i64 n, T *A, i64 lda, i64 sA, T *s, i64 lds, T *U, i64 ldu, i64 sU, T *V,
               i64 ldv, i64 sV, i64 batch) {
  if (batch <= 0) return;
  launch_svd<T>(n, kGeneral, A, lda, sA, s, lds, U, ldu, sU, V, ldv, sV, batch, nullptr);
}

template <typename T>
void eig_psd_small(i64 n, const T *A, i64 lda, i64 sA, T *s, i64 lds, T *U, i64 ldu, i64 sU,
                   i64 batch) {
  if (batch <= 0) return;
  launch_svd<T>(n, kPsd, A, lda, sA, s, lds, U, ldu, sU, (T *)nullptr, 0, 0, batch, nullptr);
}

template <typename T>
void syev_small(i64 n, const T *A, i64 lda, T *w, T *Z, i64 ldz) {
  DBuf<T> sig(n), usrt(n * n), shift(1);
  launch_svd<T>(n, kSymmetric, A, lda, 0, sig.get(), n, usrt.get(), n, 0, nullptr, 0, 0, 1, shift.get());
  hipLaunchKernelGGL(syev_finish_kernel<T>, dim3(ceil_div(n * n, 256)), dim3(256), 0,
                     ctx().stream, (int)n, (const T *)sig.get(), (const T *)shift.get(),
                     (const T *)usrt.get(), w, Z, ldz);
  LAUNCH_CHECK();
}

template void svd_small<double>(i64, double *, i64, i64, double *, i64, double *, i64, i64,
                                double *, i64, i64, i64);
template void svd_small<float>(i64, float *, i64, i64, float *, i64, float *, i64, i64, float *,
                               i64, i64, i64);
template void eig_psd_small<double>(i64, const double *, i64, i64, double *, i64, double *, i64, i64,
                                    i64);
template void eig_psd_small<float>(i64, const float *, i64, i64, float *, i64, float *, i64, i64, i64);
template void syev_small<double>(i64, const double *, i64, double *, double *, i64);
template void syev_small<float>(i64, const float *, i64, float *, float *, i64);

}  // namespace isvd
