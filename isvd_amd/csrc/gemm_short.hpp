// C (m x n) = alpha A^T B + beta C with a short K (at most 64) and a large C, both operands
// K-contiguous: the gradient dA = Pt^T Rt of a tall matrix.  Included by gemm.hip.
//
// With K <= 64 an element of C costs at most 2 K FLOP against one store: writing C bounds the product.
// Tiles through LDS spend their time on filling LDS for a handful of K steps and on the barriers
// around them.  Here a wave keeps 16 MT rows of A^T for the whole of K in registers and walks over
// columns, 16 at a time: the next group's B (one 16-byte load per lane and 16 or 8 K values) is in
// flight under the products, a lane stores four consecutive rows at once, and the four waves of a
// workgroup lie side by side in the rows (up to 256 contiguous ones per column) as far as there are
// rows.  65536 x 8192 FP32, K = 48: 1048 -> 714 us (3.0 TB/s written); one workgroup per CU with
// long strips of columns writes fastest (two 743 us, eight 860).
#pragma once

namespace isvd {

namespace shortk {
constexpr int NT = 256;
template <typename T>
struct Traits {
  static constexpr int V = 16 / sizeof(T), STEP = 4 * V;  // K values per vector and lane quadruple
};
}  // namespace shortk

// KQ = ceil(K / STEP) vectors per lane; wr of the four waves lie side by side in the rows, the others
// in the columns, of which a workgroup has `cols` (a multiple of 16).
template <typename T, int MT, int KQ>
__global__ __launch_bounds__(shortk::NT, 2) void gemm_short_kernel(GemmArgs<T> g, int wr, i64 cols) {
  using X = shortk::Traits<T>;
  constexpr int V = X::V, STEP = X::STEP;
  typedef T vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));
  typedef T out __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  using acc_t = typename Mfma<T>::acc_t;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lk = lane >> 4, K = (int)g.k;
  const T *__restrict__ A = g.A + (i64)blockIdx.y * g.sA;
  const T *__restrict__ B = g.B + (i64)blockIdx.y * g.sB;
  T *__restrict__ C = g.C + (i64)blockIdx.y * g.sC;
  // workgroups that write the same columns next to each other on one XCD
  constexpr i64 kXcd = 8;
  i64 pid = blockIdx.x;
  {
    const i64 total = gridDim.x, xcd = pid % kXcd, local = pid / kXcd;
    const i64 per = total / kXcd, rem = total % kXcd;
    pid = (xcd < rem) ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
  }
  const i64 panels = ((g.m + 16 * MT - 1) / (16 * MT) + wr - 1) / wr;
  const i64 r0 = (pid % panels * wr + wave % wr) * 16 * MT;
  const i64 c00 = pid / panels * cols, cbeg = c00 + 16 * (wave / wr);
  const i64 cend = c00 + cols < g.n ? c00 + cols : g.n;
  const int stride = 16 * (4 / wr);
  if (r0 >= g.m || cbeg >= cend) return;

  // Vector q of a lane starts at K index STEP q + V lk, or early enough to end at K: values that
  // another vector holds too count as zero in both operands.
  auto start = [&](int q) {
    const int k = STEP * q + V * lk;
    return k < K - V ? k : K - V;
  };
  auto own = [&](int q, int v) { return start(q) + v >= STEP * q + V * lk; };
  // row of the tile that instruction row lr stands for: a lane's four results are consecutive rows
  const int arow = sizeof(T) == 8 ? 4 * (lr & 3) + (lr >> 2) : lr;
  T a[MT][KQ][V];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const i64 r = r0 + 16 * t + arow;
    const T *p = A + (r < g.m ? r : g.m - 1) * g.lda;
#pragma unroll
    for (int q = 0; q < KQ; ++q) {
      const vec x = *reinterpret_cast<const vec *>(p + start(q));
#pragma unroll
      for (int v = 0; v < V; ++v) a[t][q][v] = own(q, v) ? x[v] : T(0);
    }
  }
  auto load = [&](i64 c0, vec (&b)[KQ]) {
    const i64 c = c0 + lr;
    const T *p = B + (c < g.n ? c : g.n - 1) * g.ldb;
#pragma unroll
    for (int q = 0; q < KQ; ++q) b[q] = *reinterpret_cast<const vec *>(p + start(q));
  };
  const bool whole = r0 + 16 * MT <= g.m;
  auto group = [&](i64 c0, const vec (&b)[KQ]) {
    acc_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < KQ; ++q)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const T x = STEP * (q + 1) <= KQ * STEP - 16 || own(q, v) ? b[q][v] : T(0);
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = Mfma<T>::run(a[t][q][v], x, acc[t]);
      }
    const i64 c = c0 + lr;
    if (c >= cend) return;
    T *p = C + c * g.ldc + r0 + 4 * lk;
    if (whole) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        out x = *reinterpret_cast<const out *>(&acc[t]) * g.alpha;
        if (g.beta != T(0)) x += *reinterpret_cast<const out *>(p + 16 * t) * g.beta;
        *reinterpret_cast<out *>(p + 16 * t) = x;
      }
      return;
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (r0 + 16 * t + 4 * lk + e >= g.m) continue;
        T v = g.alpha * acc[t][e];
        if (g.beta != T(0)) v += g.beta * p[16 * t + e];
        p[16 * t + e] = v;
      }
  };
  vec b0[KQ], b1[KQ];
  load(cbeg, b0);
  for (i64 c = cbeg; c < cend; c += 2 * stride) {
    load(c + stride, b1);
    __builtin_amdgcn_sched_barrier(0);
    group(c, b0);
    load(c + 2 * stride, b0);
    __builtin_amdgcn_sched_barrier(0);
    if (c + stride < cend) group(c + stride, b1);
  }
}

}  // namespace isvd
