// C (m x n) = alpha A op(B) + beta C with the operands straight from global memory in the registers
// that the matrix cores read them from: the sketch, the Gram product M = Y Y^T, the projection and the
// adjoint's products with A.  Included by gemm.hip.
//
// A tile that passes through registers, LDS and two barriers per 16 K values keeps the matrix cores
// or the memory waiting, and tiles of 128 x 256 leave ragged sizes half empty.  Here a wave owns 16 MT
// rows by 16 V E columns (V = 2 doubles or 4 floats, a 16-byte load) over one K chunk and waits for no
// other; a workgroup's four waves lie side by side and share A through the L1:
//   op(B) N-contiguous: a lane's vector holds V consecutive columns at one K index, so that the
//     16 lanes of a row group read 16 V consecutive columns; component e is column tile e, whose
//     column i is column V i + e of the block.
//   op(B) K-contiguous: a lane's vector holds V consecutive K indices of one column; component h
//     goes to instruction h, whose lane group s then stands for K index V s + h.
// op(A) has its rows contiguous (MT rows per lane in one load: row MT i + t is row i of row tile t)
// and follows whichever K index the B vector implies.  Two groups of loads alternate, one in flight
// under the other's products; chunks of K are summed by splitk_reduce_kernel.  No alignment is asked
// for, and rows are cut at multiples of 16.
//
// m <= 64 (E = 1) is bound by reading B once (16 m / 8 = 12 FLOP/B at m = 48 FP64, against a ridge of
// 15).  With a 65536 x 8192 B (64 x 64 tiles through LDS -> here): FP32 m = 32 852 -> 388 us
// K-contiguous, 841 -> 346 us N-contiguous (6.2 TB/s); FP32 m = 64 868 -> 544; FP64 m = 16 1400 ->
// 721 us (6.0 TB/s), m = 48 1574 -> 1087 / 1421 -> 940, m = 64 1600 -> 1158.  The groups must cover
// whole 128-byte lines (half lines: 530 us instead of 405), and one workgroup per CU is enough (256:
// 388 us, 1024: 536 us, for the sake of fewer partials).  Small B, short K and the number of chunks:
// stream_plan.
//
// Larger m is bound by the matrix cores and, before them, by the L1: a 64 x 64 FP32 tile takes 16
// bytes per cycle and CU from it and stops at 80 TFLOP/s, 64 x 128 (E = 2, 128 accumulators, whole
// lines in flight: one wave per SIMD) reaches 134.  FP64 needs half of that: 64 x 32 tiles, two waves
// per SIMD, and 64 x 64 for the largest.  Products before (128 x 256 tiles through LDS, filled by
// direct loads where alignment let them) -> here, one after the other with nothing else on the card:
// FP64 131072 x 16384 x 4096 252.7 -> 241.6 ms (72.8 TFLOP/s), 8192 x 2048 x 512 309 -> 249 us,
// 10007 x 3001 x 517 900 -> 545 us, Gram of 10007 x 517 215 -> 87 us; FP32 65536 x 8192 x 512 5127 ->
// 4058 us (135 TFLOP/s), 16384 x 4096 x 512 687 -> 533 us, 10007 x 3001 x 517 503 -> 304 us.  As the
// first large kernel of a whole call they take longer: 610 us for 10007 x 3001 x 517 FP64, FP32 4731
// (116 TFLOP/s) and 592 us.
#pragma once

namespace isvd {

namespace stream {
constexpr int NT = 256;  // four waves of 16 V columns each
template <typename T>
struct Traits {
  static constexpr int V = 16 / sizeof(T);
  static constexpr int COLS = 16 * V * (NT / 64);
  static constexpr int STEP = 4 * V;              // K values per step
  // steps requested together: whole 128-byte lines, but one step where the accumulators of two FP64
  // strips leave no room for two and the matrix cores bound the product anyway
  static constexpr int unroll(int E) { return sizeof(T) == 8 && E == 2 ? 1 : 2; }
  static constexpr int waves(int E) { return sizeof(T) == 4 && E == 2 ? 1 : 2; }  // per SIMD
};
// row blocks of `rows` rows that touch the upper triangle in column strip cb of `cols` columns
__host__ __device__ inline i64 upper_blocks(i64 cb, i64 rows, i64 cols, i64 rblocks) {
  const i64 c = ((cb + 1) * cols + rows - 1) / rows;
  return c < rblocks ? c : rblocks;
}
// vectors at element alignment (global memory takes 4-byte aligned wide loads)
template <typename T, int N>
struct Vec {
  typedef T type __attribute__((ext_vector_type(N), aligned(sizeof(T))));
};
// N consecutive values and nothing past them (a vector of three would be read as one of four)
template <typename T, int N>
__device__ __forceinline__ void load_values(const T *p, T (&v)[N]) {
  if constexpr (N == 2 || N == 4) {
    const typename Vec<T, N>::type x = *reinterpret_cast<const typename Vec<T, N>::type *>(p);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = x[i];
  } else if constexpr (N == 3) {
    const typename Vec<T, 2>::type x = *reinterpret_cast<const typename Vec<T, 2>::type *>(p);
    v[0] = x[0];
    v[1] = x[1];
    v[2] = p[2];
  } else {
    v[0] = p[0];
  }
}
}  // namespace stream

template <typename T, bool KB, int MT, int E>
__global__ __launch_bounds__(stream::NT, (stream::Traits<T>::waves(E))) void gemm_stream_kernel(
    GemmArgs<T> g) {
  using namespace stream;
  using X = Traits<T>;
  constexpr int V = X::V, U = X::unroll(E), STEP = X::STEP, CT = V * E;
  typedef typename Vec<T, V>::type bvec;
  typedef T avec[MT];
  using acc_t = typename Mfma<T>::acc_t;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int batch_id = blockIdx.y / g.ksplit, ks = blockIdx.y % g.ksplit;
  const i64 kbeg = (i64)ks * g.kchunk;
  const i64 kend = kbeg + g.kchunk < g.k ? kbeg + g.kchunk : g.k;
  const T *__restrict__ A = g.A + (i64)batch_id * g.sA;
  const T *__restrict__ B = g.B + (i64)batch_id * g.sB;
  // Row blocks in groups of group_m; within a group the column strips in turn, and the group's
  // blocks of one strip (which read the same part of B) next to each other on one XCD.
  i64 rb, cb;
  {
    constexpr i64 kXcd = 8;
    i64 pid = blockIdx.x;
    const i64 total = gridDim.x, xcd = pid % kXcd, local = pid / kXcd;
    const i64 per = total / kXcd, rem = total % kXcd;
    pid = (xcd < rem) ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
    const i64 rblocks = (g.m + 16 * MT - 1) / (16 * MT);
    if (g.upper) {  // the blocks that touch the upper triangle, strip by strip
      cb = 0;
      for (;;) {
        const i64 c = upper_blocks(cb, 16 * MT, X::COLS * E, rblocks);
        if (pid < c) break;
        pid -= c;
        ++cb;
      }
      rb = pid;
    } else {
      const i64 strips = (g.n + X::COLS * E - 1) / (X::COLS * E);
      const i64 first = pid / (g.group_m * strips) * g.group_m;
      const i64 in = pid % (g.group_m * strips);
      const i64 gsz = rblocks - first < g.group_m ? rblocks - first : g.group_m;
      rb = first + in % gsz;
      cb = in / gsz;
    }
  }
  const i64 r0 = rb * 16 * MT;
  const int mrows = (int)(g.m - r0 < 16 * MT ? g.m - r0 : 16 * MT);
  A += r0;
  const i64 n0 = cb * (X::COLS * E) + wave * 16 * CT;
  if (n0 >= g.n) return;

  // this lane's columns: KB: tile e at n0 + 16 e + lr; else V consecutive ones from cvec (the last
  // vector starts early where it would pass column n: its first columns are then another lane's).
  // Loads take a uniform base per step and these 32-bit byte offsets.
  i64 cnom[E], cvec[E];
  unsigned boff[CT];
  const i64 nb = KB || n0 <= g.n - V ? n0 : g.n - V;
#pragma unroll
  for (int x = 0; x < E; ++x) {
    cnom[x] = n0 + 16 * V * x + V * lr;
    cvec[x] = cnom[x] <= g.n - V ? cnom[x] : g.n - V;
  }
#pragma unroll
  for (int e = 0; e < CT; ++e) {
    const i64 c = n0 + 16 * e + lr < g.n ? n0 + 16 * e + lr : g.n - 1;
    boff[e] = (unsigned)(sizeof(T) * (KB ? (c - n0) * g.ldb + V * lk
                                         : cvec[e / V] - nb + lk * g.ldb));
  }
  // Rows: the last vector of the block starts early where it would pass row m (rows that it has in
  // common with the one before are not stored twice).  With fewer rows than a vector, the rest of it
  // comes from the next column of A, and K's last value, where there is none, from the checked rest.
  const bool short_rows = mrows < MT;
  auto row_start = [&](int i) {
    const int r = MT * i < mrows - MT ? MT * i : mrows - MT;
    return r > 0 ? r : 0;
  };
  const int arow = row_start(lr);
  const unsigned aoff = (unsigned)(sizeof(T) * (arow + (KB ? V * lk : lk) * g.lda));

  acc_t acc[MT][CT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int e = 0; e < CT; ++e) acc[t][e] = acc_t{0, 0, 0, 0};

  // K index of instruction h in the step at k0
  auto kof = [&](i64 k0, int h) { return KB ? k0 + V * lk + h : k0 + 4 * h + lk; };
  auto load = [&](i64 k0, int h, avec (&a)[V], bvec (&b)[CT]) {
    const char *bb = reinterpret_cast<const char *>(KB ? B + nb * g.ldb + k0
                                                       : B + nb + (k0 + 4 * h) * g.ldb);
#pragma unroll
    for (int x = 0; x < E; ++x)
      b[V * x + h] = *reinterpret_cast<const bvec *>(bb + boff[V * x + h]);
    const char *ab = reinterpret_cast<const char *>(A + (k0 + (KB ? h : 4 * h)) * g.lda);
    load_values<T, MT>(reinterpret_cast<const T *>(ab + aoff), a[h]);
  };
  auto mma = [&](const avec (&a)[V], const bvec (&b)[CT]) {
#pragma unroll
    for (int h = 0; h < V; ++h)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < CT; ++e)
          acc[t][e] = Mfma<T>::run(a[h][t], KB ? b[e][h] : b[e / V * V + h][e % V],
                                   acc[t][e]);
  };
  // whole groups of U steps, all inside the chunk and clear of the last column of A
  const i64 last = kend < g.k || !short_rows ? kend : g.k - 1;
  const i64 groups = last > kbeg ? (last - kbeg) / (U * STEP) : 0;
  avec a0[U][V], a1[U][V];
  bvec b0[U][CT], b1[U][CT];
  auto load_group = [&](i64 q, avec (&a)[U][V], bvec (&b)[U][CT]) {
#pragma unroll
    for (int h = 0; h < V; ++h)
#pragma unroll
      for (int u = 0; u < U; ++u) load(kbeg + (q * U + u) * STEP, h, a[u], b[u]);
  };
  auto mma_group = [&](const avec (&a)[U][V], const bvec (&b)[U][CT]) {
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
    T a[V][MT], b[V][CT];
#pragma unroll
    for (int h = 0; h < V; ++h) {
      const i64 kc = kof(k0, h) < kend ? kof(k0, h) : kend - 1;
#pragma unroll
      for (int t = 0; t < MT; ++t)
        a[h][t] = A[(arow + t < mrows ? arow + t : mrows - 1) + kc * g.lda];
#pragma unroll
      for (int e = 0; e < CT; ++e) {
        const i64 c = KB ? (n0 + 16 * e + lr < g.n ? n0 + 16 * e + lr : g.n - 1)
                         : cvec[e / V] + e % V;
        b[h][e] = KB ? B[c * g.ldb + kc] : B[c + kc * g.ldb];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < V; ++h) {
      const bool in = kof(k0, h) < kend;
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < CT; ++e)
          acc[t][e] = Mfma<T>::run(in ? a[h][t] : T(0), in ? b[h][e] : T(0), acc[t][e]);
    }
  }

  // row row_start(i) + t, i = Mfma row; column as above
  const bool split = g.ksplit > 1;
  T *C = split ? g.W + ((i64)batch_id * g.ksplit + ks) * g.m * g.n : g.C + (i64)batch_id * g.sC;
  const i64 ldc = split ? g.m : g.ldc;
#pragma unroll
  for (int e = 0; e < CT; ++e) {
    const i64 c = KB ? n0 + 16 * e + lr : cvec[e / V] + e % V;
    if (c >= g.n || (!KB && c < cnom[e / V])) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int i = Mfma<T>::row(lane, q), rl = row_start(i) + t;
        if (rl >= mrows || rl < MT * i) continue;
        const i64 r = r0 + rl;
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
