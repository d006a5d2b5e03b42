// The two products of an orthogonalization with the m x l row-major blocks Y_b (l <= 128, side by
// side in one row, so row stride ldy and block stride sY): the Gram matrices W_b = Y_b^T Y_b and
// Z_b = Y_b R_b^-1 with upper triangular R_b^-1.
//
// A row of Y_b is both operands of the Gram product and the whole reduction of the other, so both
// read Y exactly once, straight from global memory into the registers the matrix cores take it
// from; no LDS, no barriers, each wave on rows of its own.
//   Gram: with lane group g = lane / 16 on row k + g and lane % 16 on a column, one register per 16
//     columns is the A and the B operand at once.  A wave keeps the whole upper triangle of W_b (36
//     tiles at l = 128: 144 registers in FP32, 288 in FP64) over its rows; the tiles below the
//     diagonal (44 % of them at l = 128) are not computed.
//   Y R^-1: the tiles of R^-1 on and above the diagonal stay in registers (as many), a wave reads
//     16 rows of Y in 16-byte loads, each replaced by the next rows' as soon as it is used up.
// On 128 x 128 tiles through LDS both took Y through it twice and computed all of W_b and all of
// R^-1's zeros.  131072 x (32 blocks of 128), before -> here: Gram FP32 1546 -> 779 us, FP64 3140 ->
// 1244 us (62 TFLOP/s: its matrix instructions bound it); Y R^-1 FP32 1605 -> 1231 us, FP64 3201 ->
// 1693 us (5.1 TB/s, read and written).  16384 x (16 blocks of 32) FP32: Gram 33 -> 9.1 us, Y R^-1
// 25 -> 14.5 us; 10007 x (11 blocks of 63) FP64: 30 -> 16.8 us and 29 -> 31 us.
#include "la.hpp"
#include "mfma.hpp"

namespace isvd {

namespace {

constexpr int kThreads = 256;  // four waves

// waves per SIMD at `regs` accumulator and operand registers
constexpr int waves_for(int regs) {
  const int w = 512 / (regs + 40);
  return w < 1 ? 1 : (w > 4 ? 4 : w);
}
// 4-row steps requested together by the Gram kernel: enough products to cover their latency
constexpr int gram_unroll(int CT) { return CT <= 2 ? 8 : (CT <= 4 ? 4 : 2); }
// waves that share a triangle: accumulators past 256 registers would spill
template <typename T, int CT>
constexpr int gram_split() {
  return (int)sizeof(T) / 4 * 2 * CT * (CT + 1) > 200 ? 2 : 1;
}
template <typename T, int CT>
constexpr int gram_waves() {
  const int w = waves_for((int)sizeof(T) / 4 * (2 * CT * (CT + 1) / gram_split<T, CT>() +
                                                2 * gram_unroll(CT) * CT));
  return CT <= 2 && sizeof(T) == 8 ? 3 : w;  // 48 KB of LDS
}
template <typename T, int CT>
constexpr int apply_waves() {
  return waves_for((int)sizeof(T) / 4 * (2 * CT * (CT + 1) + 8 * CT));
}

// Rows blockIdx.x * chunk .. + chunk of block blockIdx.y: partial upper triangle of its Gram, tile
// (i, j) at number i + j (j + 1) / 2, element q * 64 + lane (the four waves' sums in fixed order).
template <typename T, int CT>
__global__ __launch_bounds__(kThreads, (gram_waves<T, CT>())) void gram_rows_kernel(
    int l, i64 m, i64 chunk, const T *__restrict__ Y, i64 ldy, i64 sY, T *__restrict__ P) {
  constexpr int U = gram_unroll(CT), TILES = CT * (CT + 1) / 2, STEP = 4 * U;
  constexpr int SPLIT = gram_split<T, CT>(), NACC = TILES / SPLIT, SLOTS = 4 / SPLIT;
  static_assert(TILES % SPLIT == 0, "the sharing waves have equal parts");
  constexpr int TB = 6;  // accumulators summed over the waves per round
  using acc_t = typename Mfma<T>::acc_t;
  __shared__ T red[4][TB][256];
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // wave `part` of those that share a triangle has its tiles SPLIT a + part; waves of one slot
  // have the same rows
  const int part = wave % SPLIT, slot = wave / SPLIT;
  const i64 beg = blockIdx.x * chunk, end = beg + chunk < m ? beg + chunk : m;
  // columns past l (of the last tile only) are read from column l - 1: their sums are not used
  const int clast = 16 * (CT - 1) + lr < l ? 16 * (CT - 1) + lr : l - 1;
  const T *Yb = Y + (i64)blockIdx.y * sY;

  acc_t acc[NACC];
#pragma unroll
  for (int q = 0; q < NACC; ++q) acc[q] = acc_t{0, 0, 0, 0};
  typedef T Group[U][CT];
  auto load = [&](i64 row, Group &x) {
    const T *p = Yb + (row + lk) * ldy;
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int c = 0; c < CT - 1; ++c) x[u][c] = p[16 * c + lr];
      x[u][CT - 1] = p[clast];
      p += 4 * ldy;
    }
  };
  // whole groups of STEP rows, dealt to the slots in turn; the loads are unconditional and stay in
  // front of the products of the group before.  Then the rest, four rows per slot at a time, zeros
  // past the end.
  const i64 groups = (end - beg) / STEP;
  const i64 mine = groups > slot ? (groups - slot + SLOTS - 1) / SLOTS : 0;
  auto row_of = [&](i64 q) { return beg + (SLOTS * q + slot) * STEP; };
  auto run = [&](auto part_c) {
    constexpr int PART = decltype(part_c)::value;
    auto mma = [&](const T (&x)[CT]) {
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int i = 0; i <= j; ++i) {
          const int q = i + j * (j + 1) / 2;
          if (q % SPLIT == PART) acc[q / SPLIT] = Mfma<T>::run(x[i], x[j], acc[q / SPLIT]);
        }
    };
    auto mma_group = [&](const Group &x) {
#pragma unroll
      for (int u = 0; u < U; ++u) mma(x[u]);
    };
    if (mine > 0) {
      Group x0, x1;
      load(row_of(0), x0);
      for (i64 q = 0; q + 1 < mine; q += 2) {
        load(row_of(q + 1), x1);
        __builtin_amdgcn_sched_barrier(0);
        mma_group(x0);
        load(row_of(q + 2 < mine ? q + 2 : q + 1), x0);
        __builtin_amdgcn_sched_barrier(0);
        mma_group(x1);
      }
      if (mine & 1) mma_group(x0);
    }
    for (i64 k0 = beg + groups * STEP + 4 * slot; k0 < end; k0 += 4 * SLOTS) {
      const i64 k = k0 + lk;
      const bool in = k < end;
      const T *p = Yb + (in ? k : end - 1) * ldy;
      T x[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const T v = p[c < CT - 1 ? 16 * c + lr : clast];
        x[c] = in ? v : T(0);
      }
      mma(x);
    }
  };
  if (SPLIT == 1 || part == 0) run(std::integral_constant<int, 0>{});
  else run(std::integral_constant<int, SPLIT - 1>{});

  T *Pb = P + ((i64)blockIdx.y * gridDim.x + blockIdx.x) * TILES * 256;
#pragma unroll
  for (int a0 = 0; a0 < NACC; a0 += TB) {
    if (a0) __syncthreads();
#pragma unroll
    for (int a = a0; a < NACC && a < a0 + TB; ++a)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[wave][a - a0][e * 64 + lane] = acc[a][e];
    __syncthreads();
#pragma unroll
    for (int a = a0; a < NACC && a < a0 + TB; ++a)
#pragma unroll
      for (int h = 0; h < SPLIT; ++h) {
        T v = red[h][a - a0][t];
#pragma unroll
        for (int w = h + SPLIT; w < 4; w += SPLIT) v += red[w][a - a0][t];
        Pb[(SPLIT * a + h) * 256 + t] = v;
      }
  }
}

// W (l x l per block, dense) := the sum of a block's partial triangles, mirrored
template <typename T>
__global__ __launch_bounds__(kThreads) void gram_sum_kernel(int l, int slabs, int tiles,
                                                            const T *__restrict__ P,
                                                            T *__restrict__ W) {
  const int t = threadIdx.x, lane = t & 63;
  int j = 0, i = blockIdx.x;
  while (i > j) i -= ++j;
  const T *p = P + ((i64)blockIdx.y * slabs * tiles + blockIdx.x) * 256 + t;
  T s = T(0);
#pragma unroll 8
  for (int q = 0; q < slabs; ++q) s += p[(i64)q * tiles * 256];
  const int r = 16 * i + Mfma<T>::row(lane, t >> 6), c = 16 * j + (lane & 15);
  if (r >= l || c >= l) return;
  T *Wb = W + (i64)blockIdx.y * l * l;
  Wb[r + (i64)c * l] = s;
  if (i != j) Wb[c + (i64)r * l] = s;
}

// The same for two different blocks, W_b = X_b^T Y_b (r x l): every tile of the product is computed.
// On 64 x 64 tiles with K cut in 64 parts the 16 rows of K per step came through LDS, 32 x 32 x 65536
// FP32 in 51 us and 17 us of summation; here 7.1 and 4.5 us.
// 16 C x 16 C of them per workgroup (blockIdx.z: which), partial sums in 256-element tiles, tile
// (i, j) of sub-block z at number z C^2 + i + C j.
template <typename T, int C>
__global__ __launch_bounds__(kThreads, 2) void cross_rows_kernel(int r, int l, i64 m, i64 chunk,
                                                                 const T *__restrict__ X, i64 ldx,
                                                                 i64 sX, const T *__restrict__ Y,
                                                                 i64 ldy, i64 sY,
                                                                 T *__restrict__ P) {
  constexpr int U = C <= 2 ? 4 : 2, TILES = C * C, STEP = 4 * U;
  constexpr int TB = 4;  // tiles summed over the waves per round
  using acc_t = typename Mfma<T>::acc_t;
  __shared__ T red[4][TB][256];
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const i64 beg = blockIdx.x * chunk, end = beg + chunk < m ? beg + chunk : m;
  const int nbr = (r + 16 * C - 1) / (16 * C);
  const int r0 = (blockIdx.z % nbr) * 16 * C, l0 = (blockIdx.z / nbr) * 16 * C;
  const T *Xb = X + (i64)blockIdx.y * sX, *Yb = Y + (i64)blockIdx.y * sY;
  int xc[C], yc[C];  // columns past the block are read from its last one: their sums are not used
#pragma unroll
  for (int c = 0; c < C; ++c) {
    xc[c] = r0 + 16 * c + lr < r ? r0 + 16 * c + lr : r - 1;
    yc[c] = l0 + 16 * c + lr < l ? l0 + 16 * c + lr : l - 1;
  }
  acc_t acc[TILES];
#pragma unroll
  for (int q = 0; q < TILES; ++q) acc[q] = acc_t{0, 0, 0, 0};
  auto mma = [&](const T (&x)[C], const T (&y)[C]) {
#pragma unroll
    for (int j = 0; j < C; ++j)
#pragma unroll
      for (int i = 0; i < C; ++i) acc[i + C * j] = Mfma<T>::run(x[i], y[j], acc[i + C * j]);
  };
  struct Group {
    T x[U][C], y[U][C];
  };
  auto load = [&](i64 row, Group &v) {
    const T *p = Xb + (row + lk) * ldx, *q = Yb + (row + lk) * ldy;
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        v.x[u][c] = p[xc[c]];
        v.y[u][c] = q[yc[c]];
      }
      p += 4 * ldx;
      q += 4 * ldy;
    }
  };
  auto mma_group = [&](const Group &v) {
#pragma unroll
    for (int u = 0; u < U; ++u) mma(v.x[u], v.y[u]);
  };
  const i64 groups = (end - beg) / STEP;
  const i64 mine = groups > wave ? (groups - wave + 3) / 4 : 0;
  auto row_of = [&](i64 q) { return beg + (4 * q + wave) * STEP; };
  if (mine > 0) {
    Group v0, v1;
    load(row_of(0), v0);
    for (i64 q = 0; q + 1 < mine; q += 2) {
      load(row_of(q + 1), v1);
      __builtin_amdgcn_sched_barrier(0);
      mma_group(v0);
      load(row_of(q + 2 < mine ? q + 2 : q + 1), v0);
      __builtin_amdgcn_sched_barrier(0);
      mma_group(v1);
    }
    if (mine & 1) mma_group(v0);
  }
  for (i64 k0 = beg + groups * STEP + 4 * wave; k0 < end; k0 += 16) {
    const i64 k = k0 + lk, kc = k < end ? k : end - 1;
    T x[C], y[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const T xv = Xb[kc * ldx + xc[c]], yv = Yb[kc * ldy + yc[c]];
      x[c] = k < end ? xv : T(0);
      y[c] = k < end ? yv : T(0);
    }
    mma(x, y);
  }
  T *Pb = P + (((i64)blockIdx.y * gridDim.x + blockIdx.x) * gridDim.z + blockIdx.z) * TILES * 256;
#pragma unroll
  for (int q0 = 0; q0 < TILES; q0 += TB) {
    if (q0) __syncthreads();
#pragma unroll
    for (int q = q0; q < TILES && q < q0 + TB; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[wave][q - q0][e * 64 + lane] = acc[q][e];
    __syncthreads();
#pragma unroll
    for (int q = q0; q < TILES && q < q0 + TB; ++q)
      Pb[q * 256 + t] = (red[0][q - q0][t] + red[1][q - q0][t]) +
                        (red[2][q - q0][t] + red[3][q - q0][t]);
  }
}

// W_b := alpha * the sum of its partial sums + beta W_b
template <typename T, int C>
__global__ __launch_bounds__(4 * kThreads) void cross_sum_kernel(int r, int l, int slabs, int tiles,
                                                                 const T *__restrict__ P, T alpha,
                                                                 T beta, T *__restrict__ W,
                                                                 i64 ldw, i64 sW) {
  __shared__ T red[3][kThreads];
  const int t = threadIdx.x % kThreads, part = threadIdx.x / kThreads, lane = t & 63;
  const int z = blockIdx.x / (C * C), q = blockIdx.x % (C * C), nbr = (r + 16 * C - 1) / (16 * C);
  const T *p = P + ((i64)blockIdx.y * slabs * tiles + blockIdx.x) * 256 + t;
  T s = T(0);
#pragma unroll 8
  for (int k = part; k < slabs; k += 4) s += p[(i64)k * tiles * 256];
  if (part > 0) red[part - 1][t] = s;
  __syncthreads();
  if (part > 0) return;
  s += red[0][t] + (red[1][t] + red[2][t]);
  const int i = (z % nbr) * 16 * C + 16 * (q % C) + Mfma<T>::row(lane, t >> 6);
  const int j = (z / nbr) * 16 * C + 16 * (q / C) + (lane & 15);
  if (i >= r || j >= l) return;
  T *w = W + (i64)blockIdx.y * sW + i + (i64)j * ldw;
  s *= alpha;
  if (beta != T(0)) s += beta * *w;
  *w = s;
}

// Z_b := Y_b X_b, X_b l x l upper triangular, dense column-major; a wave takes every nwaves-th
// group of 16 rows.
template <typename T, int CT>
__global__ __launch_bounds__(kThreads, (apply_waves<T, CT>())) void apply_upper_kernel(
    int l, i64 m, const T *__restrict__ Y, i64 ldy, i64 sY, const T *__restrict__ X,
    T *__restrict__ Z, i64 ldz, i64 sZ) {
  constexpr int V = 16 / sizeof(T), H = 4 / V, TILES = CT * (CT + 1) / 2;
  typedef T vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));
  using acc_t = typename Mfma<T>::acc_t;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const i64 id = (i64)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  const i64 nwaves = (i64)gridDim.x * (kThreads / 64), groups = (m + 15) / 16;
  if (id >= groups) return;
  const T *Yb = Y + (i64)blockIdx.y * sY, *Xb = X + (i64)blockIdx.y * l * l;
  T *Zb = Z + (i64)blockIdx.y * sZ;

  // Lane group lk's vector h of column tile c starts at column 16 c + 4 V h + V lk, or early enough
  // to end at column l: columns that another vector holds too then meet zeros of X.
  auto col_of = [&](int c, int h) {
    const int k = 16 * c + 4 * V * h + V * lk;
    return k < l - V ? k : l - V;
  };
  T x[TILES][4];
#pragma unroll
  for (int j = 0; j < CT; ++j)
#pragma unroll
    for (int c = 0; c <= j; ++c)
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int v = 0; v < V; ++v) {
          const int k = col_of(c, h) + v, n = 16 * j + lr;
          const bool in = k >= 16 * c + 4 * V * h + V * lk && k <= n && n < l;
          x[c + j * (j + 1) / 2][V * h + v] = in ? Xb[k + (i64)n * l] : T(0);
        }

  vec y[CT][H];
  auto load = [&](i64 grp, int c) {
    const i64 r = 16 * grp + lr;
    const T *p = Yb + (r < m ? r : m - 1) * ldy;
#pragma unroll
    for (int h = 0; h < H; ++h) y[c][h] = *reinterpret_cast<const vec *>(p + col_of(c, h));
  };
#pragma unroll
  for (int c = 0; c < CT; ++c) load(id, c);
  for (i64 grp = id; grp < groups; grp += nwaves) {
    const i64 next = grp + nwaves < groups ? grp + nwaves : grp;
    acc_t acc[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[j] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < CT; ++c) {
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
          for (int j = c; j < CT; ++j)
            acc[j] = Mfma<T>::run(y[c][h][v], x[c + j * (j + 1) / 2][V * h + v], acc[j]);
      load(next, c);
    }
    const i64 r0 = 16 * grp;
    T *q = Zb + r0 * ldz + lr;
    const bool clast = 16 * (CT - 1) + lr < l;
    if (r0 + 16 <= m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        T *z = q + Mfma<T>::row(lane, e) * ldz;
#pragma unroll
        for (int j = 0; j < CT - 1; ++j) z[16 * j] = acc[j][e];
        if (clast) z[16 * (CT - 1)] = acc[CT - 1][e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int rr = Mfma<T>::row(lane, e);
        T *z = q + rr * ldz;
#pragma unroll
        for (int j = 0; j < CT; ++j)
          if (r0 + rr < m && 16 * j + lr < l) z[16 * j] = acc[j][e];
      }
    }
  }
}

template <typename T, int CT>
bool launch_gram(i64 l, i64 m, const T *Y, i64 ldy, i64 sY, T *W, i64 batch) {
  constexpr int TILES = CT * (CT + 1) / 2, ROWS = 16 * gram_unroll(CT);
  // one round of the waves that fit, each with at least one group of rows
  i64 slabs = (ctx().cus * gram_waves<T, CT>() + batch - 1) / batch;
  const i64 most = (m + ROWS - 1) / ROWS;
  if (slabs > most) slabs = most;
  const size_t per = sizeof(T) * (size_t)(batch * TILES * 256), room = splitk_budget();
  if (room < per) return false;
  if ((size_t)slabs > room / per) slabs = (i64)(room / per);
  i64 chunk = (m + slabs - 1) / slabs;
  chunk = (chunk + ROWS - 1) / ROWS * ROWS;
  slabs = (m + chunk - 1) / chunk;
  T *P = static_cast<T *>(splitk_workspace(per * (size_t)slabs));
  hipLaunchKernelGGL((gram_rows_kernel<T, CT>), dim3((unsigned)slabs, (unsigned)batch),
                     dim3(kThreads), 0, ctx().stream, (int)l, m, chunk, Y, ldy, sY, P);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(gram_sum_kernel<T>, dim3(TILES, (unsigned)batch), dim3(kThreads), 0,
                     ctx().stream, (int)l, (int)slabs, TILES, (const T *)P, W);
  LAUNCH_CHECK();
  return true;
}

template <typename T, int CT>
void launch_apply(i64 l, i64 m, const T *X, const T *Y, i64 ldy, i64 sY, T *Z, i64 ldz, i64 sZ,
                  i64 batch) {
  i64 wgs = (ctx().cus * apply_waves<T, CT>() + batch - 1) / batch;
  const i64 most = ((m + 15) / 16 + 3) / 4;
  if (wgs > most) wgs = most;
  hipLaunchKernelGGL((apply_upper_kernel<T, CT>), dim3((unsigned)wgs, (unsigned)batch),
                     dim3(kThreads), 0, ctx().stream, (int)l, m, Y, ldy, sY, X, Z, ldz, sZ);
  LAUNCH_CHECK();
}

template <typename T, int C>
bool launch_cross(i64 r, i64 l, i64 m, T alpha, const T *X, i64 ldx, i64 sX, const T *Y, i64 ldy,
                  i64 sY, T beta, T *W, i64 ldw, i64 sW, i64 batch) {
  constexpr int ROWS = 16 * (C <= 2 ? 4 : 2);
  const i64 blocks = ((r + 16 * C - 1) / (16 * C)) * ((l + 16 * C - 1) / (16 * C));
  const i64 tiles = blocks * C * C;
  i64 slabs = (2 * ctx().cus + batch * blocks - 1) / (batch * blocks);
  const i64 most = (m + 2 * ROWS - 1) / (2 * ROWS);
  if (slabs > 128) slabs = 128;  // one workgroup sums a tile's parts
  if (slabs > most) slabs = most;
  const size_t per = sizeof(T) * (size_t)(batch * tiles * 256), room = splitk_budget();
  if (room < per) return false;
  if ((size_t)slabs > room / per) slabs = (i64)(room / per);
  i64 chunk = (m + slabs - 1) / slabs;
  chunk = (chunk + ROWS - 1) / ROWS * ROWS;
  slabs = (m + chunk - 1) / chunk;
  T *P = static_cast<T *>(splitk_workspace(per * (size_t)slabs));
  hipLaunchKernelGGL((cross_rows_kernel<T, C>),
                     dim3((unsigned)slabs, (unsigned)batch, (unsigned)blocks), dim3(kThreads), 0,
                     ctx().stream, (int)r, (int)l, m, chunk, X, ldx, sX, Y, ldy, sY, P);
  LAUNCH_CHECK();
  hipLaunchKernelGGL((cross_sum_kernel<T, C>), dim3((unsigned)tiles, (unsigned)batch),
                     dim3(4 * kThreads), 0, ctx().stream, (int)r, (int)l, (int)slabs, (int)tiles,
                     (const T *)P, alpha, beta, W, ldw, sW);
  LAUNCH_CHECK();
  return true;
}

// f(std::integral_constant<int, CT>) for CT = ceil(l / 16) in 1 .. 8
template <typename F>
auto by_tiles(i64 l, F f) {
  switch ((l + 15) / 16) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 5: return f(std::integral_constant<int, 5>{});
    case 6: return f(std::integral_constant<int, 6>{});
    case 7: return f(std::integral_constant<int, 7>{});
    default: return f(std::integral_constant<int, 8>{});
  }
}

}  // namespace

template <typename T>
void gram_rows(i64 l, i64 m, const T *Y, i64 ldy, i64 sY, T *W, i64 batch) {
  ISVD_CHECK(l > 0 && m > 0 && batch > 0 && ldy >= l, "gram_rows: bad arguments");
  // wider blocks, more of them than a grid's second dimension, and a scratch region without room
  // for one set of partial sums: the general product
  if (l <= 128 && batch <= 65535 &&
      by_tiles(l, [&](auto ct) {
        return launch_gram<T, decltype(ct)::value>(l, m, Y, ldy, sY, W, batch);
      }))
    return;
  gemm<T>('N', 'T', l, l, m, T(1), Y, ldy, Y, ldy, T(0), W, l, batch, sY, sY, l * l);
}

template <typename T>
bool cross_rows(i64 r, i64 l, i64 m, T alpha, const T *X, i64 ldx, i64 sX, const T *Y, i64 ldy,
                i64 sY, T beta, T *W, i64 ldw, i64 sW, i64 batch) {
  const i64 most = r > l ? r : l;
  if (most > 128 || batch > 65535) return false;
  if (most <= 16)
    return launch_cross<T, 1>(r, l, m, alpha, X, ldx, sX, Y, ldy, sY, beta, W, ldw, sW, batch);
  if (most <= 32)
    return launch_cross<T, 2>(r, l, m, alpha, X, ldx, sX, Y, ldy, sY, beta, W, ldw, sW, batch);
  if (most <= 48 || (most > 64 && most <= 96))
    return launch_cross<T, 3>(r, l, m, alpha, X, ldx, sX, Y, ldy, sY, beta, W, ldw, sW, batch);
  return launch_cross<T, 4>(r, l, m, alpha, X, ldx, sX, Y, ldy, sY, beta, W, ldw, sW, batch);
}

template <typename T>
void apply_upper(i64 l, i64 m, const T *X, const T *Y, i64 ldy, i64 sY, T *Z, i64 ldz, i64 sZ,
                 i64 batch) {
  ISVD_CHECK(l > 0 && m > 0 && batch > 0 && ldy >= l && ldz >= l, "apply_upper: bad arguments");
  if (l >= (i64)(16 / sizeof(T)) && l <= 128 && batch <= 65535) {  // at least one vector per row
    by_tiles(l, [&](auto ct) {
      launch_apply<T, decltype(ct)::value>(l, m, X, Y, ldy, sY, Z, ldz, sZ, batch);
    });
    return;
  }
  gemm<T>('T', 'N', l, m, l, T(1), X, l, Y, ldy, T(0), Z, ldz, batch, l * l, sY, sZ);
}

#define ROW_BLOCKS(T)                                                                       \
  template void gram_rows<T>(i64, i64, const T *, i64, i64, T *, i64);                      \
  template bool cross_rows<T>(i64, i64, i64, T, const T *, i64, i64, const T *, i64, i64, T, T *,   \
                              i64, i64, i64);                                                \
  template void apply_upper<T>(i64, i64, const T *, const T *, i64, i64, T *, i64, i64, i64);
ROW_BLOCKS(double)
ROW_BLOCKS(float)

}  // namespace isvd
