// C (m x n) = alpha A op(B) + beta C for few rows, m <= 64, against a large op(B) (K x n): the
// projection Z^T = Qbar^T A and the adjoint's products with A.  Included by gemm.hip.
//
// At m <= 64 the product is bound by reading B once (2 m FLOP per element: 16 m / 8 = 12 FLOP/B at
// m = 48 FP64, 16 FLOP/B at m = 32 FP32, against a ridge of 15 and 31).  The tiled kernels pass
// every tile of B through registers, LDS and two barriers per 16 K values and reach 2.5 TB/s; here B
// goes from global memory straight into the registers the matrix cores read it from, in 16-byte
// loads (V = 2 doubles or 4 floats), 8 of them in flight per wave, and no wave waits for another:
//   op(B) MN-contiguous: a lane's vector holds V consecutive columns at one K index, so that the
//     16 lanes of a row group read 16 V consecutive columns; component e is column tile e, whose
//     column i is column V i + e of the block.
//   op(B) K-contiguous: a lane's vector holds V consecutive K indices of one column; component h
//     goes to instruction h, whose lane group s then stands for K index V s + h.
// op(A) has its rows contiguous (MT rows per lane in one load: row MT i + t is row i of row tile t),
// is small enough for the caches, and follows whichever K index the B vector implies.  A wave
// computes all m rows by 16 V columns over one K chunk; chunks are summed by splitk_reduce_kernel.
//
// Measured with a 65536 x 8192 B (64 x 64 tiles -> here): FP32 m = 32 852 -> 388 us K-contiguous,
// 841 -> 346 us MN-contiguous (6.2 TB/s); FP32 m = 64 868 -> 588; FP64 m = 16 1400 -> 721 us
// (6.0 TB/s), m = 48 1574 -> 1087 / 1421 -> 940, m = 64 1600 -> 1158 (59 TFLOP/s: the matrix cores
// bound it from m = 48 on).  Two groups of 2 V vectors alternate, one in flight under the
// other's products; the groups must cover whole 128-byte lines (half lines: 530 us instead of 405),
// and one workgroup per CU is enough (256: 388 us, 1024: 536 us, for the sake of fewer partials).
#pragma once

namespace isvd {

namespace thin {
constexpr int NT = 256;  // four waves of 16 V columns each
template <typename T>
struct Traits {
  static constexpr int V = 16 / sizeof(T);
  static constexpr int COLS = 16 * V * (NT / 64);
  static constexpr int STEP = 4 * V;              // K values per step
  static constexpr int U = 2;                     // steps requested together: 128-byte lines
};
// vectors at element alignment (global memory takes 4-byte aligned wide loads)
template <typename T, int N>
struct Vec {
  typedef T type __attribute__((ext_vector_type(N), aligned(sizeof(T))));
};
template <typename T>
struct Vec<T, 1> {
  typedef T type;
};
template <typename T, int N>
__device__ __forceinline__ T at(const typename Vec<T, N>::type &v, int i) {
  if constexpr (N == 1) return v;
  else return v[i];
}
}  // namespace thin

template <typename T, bool KB, int MT>
__global__ __launch_bounds__(thin::NT, 2) void gemm_thin_kernel(GemmArgs<T> g) {
  using namespace thin;
  using X = Traits<T>;
  constexpr int V = X::V, U = X::U, STEP = X::STEP;
  typedef typename Vec<T, V>::type bvec;
  typedef typename Vec<T, MT>::type avec;
  using acc_t = typename Mfma<T>::acc_t;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int batch_id = blockIdx.y / g.ksplit, ks = blockIdx.y % g.ksplit;
  const i64 kbeg = (i64)ks * g.kchunk;
  const i64 kend = kbeg + g.kchunk < g.k ? kbeg + g.kchunk : g.k;
  const T *__restrict__ A = g.A + (i64)batch_id * g.sA;
  const T *__restrict__ B = g.B + (i64)batch_id * g.sB;
  const i64 n0 = (i64)blockIdx.x * X::COLS + wave * 16 * V;
  if (n0 >= g.n) return;

  // this lane's columns: KB: tile e at n0 + 16 e + lr; else V consecutive ones from cvec (the last
  // vector starts early where it would pass column n: its first columns are then another lane's)
  const i64 cnom = n0 + V * lr;
  const i64 cvec = cnom <= g.n - V ? cnom : g.n - V;
  i64 bcol[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const i64 c = n0 + 16 * e + lr;
    bcol[e] = (c < g.n ? c : g.n - 1) * g.ldb;
  }
  // rows past m are read from the next column of A (the last step, where there is none, is the
  // checked one); they feed only outputs that are not stored
  const int arow = MT * lr < g.m ? MT * lr : 0;

  acc_t acc[MT][V];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int e = 0; e < V; ++e) acc[t][e] = acc_t{0, 0, 0, 0};

  // K index of instruction h in the step at k0
  auto kof = [&](i64 k0, int h) { return KB ? k0 + V * lk + h : k0 + 4 * h + lk; };
  auto load = [&](i64 k0, int h, avec (&a)[V], bvec (&b)[V]) {
    if (KB) b[h] = *reinterpret_cast<const bvec *>(B + bcol[h] + k0 + V * lk);
    else b[h] = *reinterpret_cast<const bvec *>(B + cvec + kof(k0, h) * g.ldb);
    a[h] = *reinterpret_cast<const avec *>(A + arow + kof(k0, h) * g.lda);
  };
  auto mma = [&](const avec (&a)[V], const bvec (&b)[V]) {
#pragma unroll
    for (int h = 0; h < V; ++h)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < V; ++e)
          acc[t][e] = Mfma<T>::run(at<T, MT>(a[h], t), KB ? b[e][h] : b[h][e], acc[t][e]);
  };
  // whole groups of U steps, all inside the chunk and clear of the last column of A
  const i64 last = kend < g.k ? kend : g.k - 1;
  const i64 groups = last > kbeg ? (last - kbeg) / (U * STEP) : 0;
  avec a0[U][V], a1[U][V];
  bvec b0[U][V], b1[U][V];
  auto load_group = [&](i64 q, avec (&a)[U][V], bvec (&b)[U][V]) {
#pragma unroll
    for (int h = 0; h < V; ++h)
#pragma unroll
      for (int u = 0; u < U; ++u) load(kbeg + (q * U + u) * STEP, h, a[u], b[u]);
  };
  auto mma_group = [&](const avec (&a)[U][V], const bvec (&b)[U][V]) {
#pragma unroll
    for (int u = 0; u < U; ++u) mma(a[u], b[u]);
  };
  // Every load is unconditional and stays in front of the products of the group before (a branch
  // around it, or its sinking into one, makes the compiler wait for everything in flight).
  if (groups > 0) {
    load_group(0, a0, b0);
    for (i64 q = 0; q + 1 < groups; q += 2) {
      load_group(q + 1, a1, b1);
      __builtin_amdgcn_sched_barrier(0);
      mma_group(a0, b0);
      load_group(q + 2 < groups ? q + 2 : q + 1, a0, b0);
      __builtin_amdgcn_sched_barrier(0);
      mma_group(a1, b1);
    }
    if (groups & 1) mma_group(a0, b0);
  }
  // the rest of the chunk: checked, zeros past its end
  for (i64 k0 = kbeg + groups * U * STEP; k0 < kend; k0 += STEP) {
#pragma unroll
    for (int h = 0; h < V; ++h) {
      const i64 k = kof(k0, h);
      const bool in = k < kend;
      const i64 kc = in ? k : kend - 1;
      T a[MT], b[V];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int r = arow + t < g.m ? arow + t : (int)g.m - 1;
        a[t] = in ? A[r + kc * g.lda] : T(0);
      }
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const T v = KB ? B[bcol[e] + kc] : B[cvec + e + kc * g.ldb];
        b[e] = in ? v : T(0);
      }
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[t][e] = Mfma<T>::run(a[t], b[e], acc[t][e]);
    }
  }

  // row MT i + t, i = Mfma row; column as above
  const bool split = g.ksplit > 1;
  T *C = split ? g.W + ((i64)batch_id * g.ksplit + ks) * g.m * g.n : g.C + (i64)batch_id * g.sC;
  const i64 ldc = split ? g.m : g.ldc;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const i64 c = KB ? n0 + 16 * e + lr : cvec + e;
    if (c >= g.n || (!KB && c < cnom)) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int r = MT * Mfma<T>::row(lane, q) + t;
        if (r >= g.m) continue;
        T v = acc[t][e][q];
        if (!split) {
          v *= g.alpha;
          if (g.beta != T(0)) v += g.beta * C[r + c * ldc];
        }
        C[r + c * ldc] = v;
      }
  }
}

}  // namespace isvd
