// The Kolmogorov-Nagumo loop in sketch coordinates, all iterations in one launch, for small l
// (FP64 l <= 64, FP32 l <= 80: the l x l matrices of the chain fit in one workgroup's LDS) and
// Nl <= 2048.
//
// There an iteration is a few microseconds of arithmetic (G = M Bg / N is 2 Nl^2 l FLOP, the rest
// l x l and Nl x l products), and as separate launches (G on a second stream, its reduction, the
// l x l chain over workgroups, the update, the Gram) it is all launch and hand-over.  Measured per
// iteration, one launch against separate ones:
//   FP64  l = 16, Nl = 128: 8.6 / 49 us   l = 32, Nl = 512: 14 / 55 us   l = 64, Nl = 2048: 58 / 84 us
//   FP32  l = 16, Nl = 128: 7.2 / 45 us   l = 32, Nl = 512: 11 / 50 us   l = 64, Nl = 2048: 38 / 70 us
//         l = 80, Nl = 2000: 61 / 71 us;  l = 96 (Nl = 2016: 80 / 75 us) stays with separate launches
// (32 rows per workgroup instead of 16: 10-35 % slower at every size.)  What bounds it: the two
// grid barriers and the reads behind them (about 6 us), then the chain's dependent products in one
// workgroup (FP64 l = 64: about 25 us) and Bg, which every workgroup reads whole.
//
// Workgroup w of a persistent grid owns 16 rows of the state [X | B | Bg | G] (in LDS) and the
// same rows of M, and every iteration has two grid barriers, the second of them behind G:
//   - sum a share of the Gram partials of all workgroups -> [D | Dg] (device-coherent), arrive;
//   - G := M Bg / N for the own rows (M from L2, Bg as the others published it), K split over the
//     waves;
//   - the l x l chain C = f(Z), C^-1, F = C - D C^-1 in LDS, by every workgroup for itself (the
//     same instructions on the same data: the same bits, so every workgroup also takes the same
//     decision about convergence and the host is not asked);
//   - X_+, B_+, Bg_+ of the own rows, their Gram partial, Bg_+ published, arrive.
// The formulas, the series, the Newton-Schulz fallback and the step counts are those of kn_chain
// (smallla.hip), and so are the grid barrier and the exchange (agent-scope atomics without
// fences).  When Z is out of reach of both, the kernel leaves with status 1 and its state, and the
// caller does that iteration by the eigendecomposition and enters again.
#include "kn_common.hpp"
#include "kn_rule.hpp"
#include "la.hpp"

#include <type_traits>

namespace isvd {

namespace {

constexpr int kLoopWaves = 8;
constexpr int kLoopThreads = 64 * kLoopWaves;

template <typename T>
struct KnLoopArgs {
  int l, Nl, mode, resume;
  i64 maxit;       // iterations of this launch at most
  i64 it0, itmax;  // iterations done before; the caller's limit
  double tol;
  T ninv;
  const T *M;      // Nl x Nl, symmetric, ld Nl
  T *state;        // X | B | Bg | G, Nl x l each (ld Nl): in with resume, out on leaving
  T *bgpub;        // 2 x (rows x L), row by row
  T *parts;        // workgroups x 2 L^2
  T *ddg;          // D | Dg, ld L, summed and scaled by 1/N
  unsigned spins;  // polls before a wait gives up
  double *scal;    // [0] ||C - I||_F, [1] iterations done, [2] rho, [3] status, [4] timed out
  unsigned long long *bar;
  T coef[2 * kSeriesTerms];
  double rho_max[kSeriesBlocks + 1];  // [t]: the largest rho that t blocks of the series serve
};

// NT: l padded to L = 16 NT
template <typename T, int NT>
struct LoopLds {
  static constexpr int L = 16 * NT, LD = L + 1, R = kLoopRows, LDR = R + 1;
  static constexpr int SLOT = L * LD;          // one l x l matrix
  static constexpr int GRED = kLoopWaves * NT * 256;  // G's K partials, before the chain
  static constexpr int WORK = 3 * SLOT > GRED ? 3 * SLOT : GRED;
  static constexpr int STATE = 4 * L * LDR;
  static constexpr size_t bytes = sizeof(T) * (size_t)(WORK + STATE);
};

template <typename T, int NT>
__global__ __launch_bounds__(kLoopThreads) void kn_loop_kernel(KnLoopArgs<T> a) {
  using S = LoopLds<T, NT>;
  using acc_t = typename SM<T>::acc;
  constexpr int L = S::L, LD = S::LD, R = S::R, LDR = S::LDR, LL = L * L;
  constexpr int TILES = NT * NT;                                  // of an l x l matrix
  constexpr int TPW = (TILES + kLoopWaves - 1) / kLoopWaves;      // per wave
  constexpr int DPT = (LL + kLoopThreads - 1) / kLoopThreads;     // entries of D per thread
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *work = reinterpret_cast<T *>(smem_raw);
  T *s1 = work, *s2 = work + S::SLOT, *s3 = work + 2 * S::SLOT;
  T *st = work + S::WORK;  // X | B | Bg | G: column c of matrix j at st + (j L + c) LDR
  __shared__ T coef[2 * kSeriesTerms];
  __shared__ double red[kLoopWaves];
  __shared__ int ok_sh;

  int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lr = lane & 15, lk = lane >> 4;
  // the lane's indices are opaque from here on: the addresses formed from them are computed where
  // they are used, not kept in registers through the loop (which spilled 80-110 of them)
  auto opaque = [&] { asm volatile("" : "+v"(tid), "+v"(lane), "+v"(lr), "+v"(lk)); };
  const int l = a.l, Nl = a.Nl, P = gridDim.x;
  const int row0 = blockIdx.x * R;
  const i64 ldm = Nl;
  unsigned long long epoch = 0;

  if (tid < 2 * kSeriesTerms) coef[tid] = a.coef[tid];

  // ---- grid barrier, in two halves ----
  auto arrive = [&] {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    epoch += (unsigned long long)P;
    if (tid == 0)
      (void)__hip_atomic_fetch_add(a.bar + kBarCount, 1ull, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
  };
  auto wait = [&]() -> bool {  // false when it timed out here or elsewhere
    if (tid == 0) {
      int ok = 1;
      unsigned spins = 0;
      while (__hip_atomic_load(a.bar + kBarCount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
             epoch) {
        if (++spins > a.spins) {
          __hip_atomic_store(a.bar + kBarAbort, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ok = 0;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      if (__hip_atomic_load(a.bar + kBarAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ok = 0;
      ok_sh = ok;
    }
    __syncthreads();
    return ok_sh != 0;
  };

  // ---- st[dst] := M src / N on the own rows; src(k, c) at src[k lds + c], c < cmax ----
  // (transposed: op(A) rows are columns of src, its columns the own rows; M is symmetric, so its
  // rows are read as columns.)  Ends with a workgroup barrier.
  auto g_product = [&](const T *src, i64 lds, int cmax, int dst) {
    acc_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = acc_t{0, 0, 0, 0};
    const int kper = ((Nl + kLoopWaves - 1) / kLoopWaves + 3) / 4 * 4;
    const int k0 = wave * kper;
    const int k1 = k0 + kper < Nl ? k0 + kper : Nl;
    const bool mok = row0 + lr < Nl;
    const int mrow = mok ? row0 + lr : Nl - 1;
    bool cok[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) cok[t] = 16 * t + lr < cmax;
    constexpr int U = NT * sizeof(T) > 16 ? 4 : 8;  // K steps requested together
    for (int k = k0; k < k1; k += 4 * U) {
      T fa[U][NT], fb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int kk = k + 4 * u + lk;
        const i64 kc = kk < k1 ? kk : k1 - 1;
#pragma unroll
        for (int t = 0; t < NT; ++t)
          fa[u][t] = cld(src + kc * lds + (cok[t] ? 16 * t + lr : 0));
        fb[u] = a.M[kc * ldm + mrow];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = k + 4 * u + lk < k1;
#pragma unroll
        for (int t = 0; t < NT; ++t) fa[u][t] = (in && cok[t]) ? fa[u][t] : T(0);
        fb[u] = (in && mok) ? fb[u] : T(0);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = SM<T>::mfma(fa[u][t], fb[u], acc[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) work[(wave * NT + t) * 256 + g * 64 + lane] = acc[t][g];
    __syncthreads();
    constexpr int E = NT * 256;
    for (int e = tid; e < E; e += kLoopThreads) {
      T s = work[e];
#pragma unroll
      for (int w = 1; w < kLoopWaves; ++w) s += work[w * E + e];
      const int tile = e >> 8, g = (e >> 6) & 3, ln = e & 63;
      const int c = 16 * tile + SM<T>::row(ln, g), r = ln & 15;
      st[(dst * L + c) * LDR + r] = a.ninv * s;
    }
    __syncthreads();
  };

  // ---- own rows' part of [D | Dg] (transposed tiles: stores run along the columns) ----
  auto gram = [&] {
    T *mine = a.parts + (i64)blockIdx.x * 2 * LL;
    for (int job = wave; job < 2 * TILES; job += kLoopWaves) {
      const int mat = job / TILES, tile = job % TILES;
      const int ti = tile % NT, tj = tile / NT;  // D(i, j): i in B, j in B (mat 0) or Bg (1)
      acc_t acc = {0, 0, 0, 0};
      const T *pj = st + ((1 + mat) * L + 16 * tj + lr) * LDR + lk;
      const T *pi = st + (L + 16 * ti + lr) * LDR + lk;
#pragma unroll
      for (int s = 0; s < R / 4; ++s) acc = SM<T>::mfma(pj[4 * s], pi[4 * s], acc);
#pragma unroll
      for (int g = 0; g < 4; ++g)
        cst(mine + mat * LL + (16 * ti + lr) + (16 * tj + SM<T>::row(lane, g)) * L, acc[g]);
    }
  };
  // ---- Bg of the own rows, for the others ----
  auto publish = [&](int parity) {
    T *dst = a.bgpub + ((i64)parity * P * R + row0) * L;
    for (int e = tid; e < R * L; e += kLoopThreads) {
      const int r = e / L, c = e % L;
      cst(dst + e, st[(2 * L + c) * LDR + r]);
    }
  };
  auto save = [&](int j, T *dst) {
    for (int e = tid; e < R * l; e += kLoopThreads) {
      const int r = e % R, c = e / R;
      if (row0 + r < Nl) dst[row0 + r + (i64)c * Nl] = st[(j * L + c) * LDR + r];
    }
  };

  // ---- this wave's tiles of an l x l matrix: tile w + 8 u at (tm, tn) ----
  int tm[TPW], tn[TPW];
  bool live[TPW];
#pragma unroll
  for (int u = 0; u < TPW; ++u) {
    const int tile = wave + kLoopWaves * u;
    live[u] = tile < TILES;
    tm[u] = tile % NT;
    tn[u] = tile / NT;
  }
  // o := op(A) B over this wave's tiles
  auto mm = [&](const T *A, const T *B, bool ta, acc_t (&o)[TPW]) {
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      o[u] = acc_t{0, 0, 0, 0};
      if (live[u]) {
        const int row = 16 * tm[u] + lr;
        const T *pa = ta ? A + row * LD + lk : A + lk * LD + row;
        const int sa = ta ? 4 : 4 * LD;
        const T *pb = B + (16 * tn[u] + lr) * LD + lk;
#pragma unroll 4
        for (int s = 0; s < 4 * NT; ++s) o[u] = SM<T>::mfma(pa[s * sa], pb[4 * s], o[u]);
      }
    }
  };
  auto put = [&](T *dst, const acc_t (&o)[TPW]) {
#pragma unroll
    for (int u = 0; u < TPW; ++u)
      if (live[u])
#pragma unroll
        for (int g = 0; g < 4; ++g)
          dst[16 * tm[u] + SM<T>::row(lane, g) + (16 * tn[u] + lr) * LD] = o[u][g];
  };
  // delta(r, c) of this lane's entry
  auto delta = [&](int u, int g) {
    return 16 * tm[u] + SM<T>::row(lane, g) == 16 * tn[u] + lr ? T(1) : T(0);
  };
  // the sum of v over the workgroup, in a fixed order (two workgroup barriers)
  auto block_sum = [&](T v) -> double {
    double x = (double)v;
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    if (lane == 0) red[wave] = x;
    __syncthreads();
    double s = 0;
#pragma unroll
    for (int w = 0; w < kLoopWaves; ++w) s += red[w];
    __syncthreads();
    return s;
  };
  auto norm2 = [&](const acc_t (&o)[TPW]) -> T {
    T s = 0;
#pragma unroll
    for (int u = 0; u < TPW; ++u)
#pragma unroll
      for (int g = 0; g < 4; ++g) s += o[u][g] * o[u][g];  // entries past l and dead tiles are 0
    return s;
  };

  // ---- first state ----
  for (int e = tid; e < 4 * L * LDR; e += kLoopThreads) st[e] = T(0);
  __syncthreads();
  for (int e = tid; e < R * l; e += kLoopThreads) {
    const int r = e % R, c = e / R;
    const int gr = row0 + r;
    if (gr < Nl) {
      if (a.resume) {
        for (int j = 0; j < 3; ++j)
          st[(j * L + c) * LDR + r] = a.state[(i64)j * Nl * l + gr + (i64)c * Nl];
      } else {
        // X := [I; 0], B := M [I; 0]
        st[c * LDR + r] = gr == c ? T(1) : T(0);
        st[(L + c) * LDR + r] = a.M[gr + (i64)c * ldm];
      }
    }
  }
  __syncthreads();
  if (!a.resume) g_product(a.M, ldm, l, 2);  // Bg := M B / N (M symmetric: B's rows are M's)
  gram();
  publish(0);
  int parity = 0;

  int status = 3;
  double err = 0, rho = 0;
  i64 done = 0;
  while (done < a.maxit) {
    opaque();
    arrive();
    if (!wait()) { status = 2; break; }
    // [D | Dg]: this workgroup's share of the entries, each the sum of all partials in order
    {
      const int cnt = (2 * LL + P - 1) / P, e0 = blockIdx.x * cnt;
      int tpe = 1;
      while (tpe < 64 && 2 * tpe * cnt <= kLoopThreads && 2 * tpe <= P) tpe *= 2;
      const int q = tid % tpe, per = (P + tpe - 1) / tpe;
      for (int i0 = 0; i0 < cnt; i0 += kLoopThreads / tpe) {
        const int e = e0 + i0 + tid / tpe;
        const bool in = i0 + tid / tpe < cnt && e < 2 * LL;
        T s = 0;
        if (in) {
          const T *src = a.parts + e;
          int w = q * per;
          const int w1 = w + per < P ? w + per : P;
          for (; w + 4 <= w1; w += 4) {
            const T v0 = cld(src + (i64)w * 2 * LL), v1 = cld(src + (i64)(w + 1) * 2 * LL);
            const T v2 = cld(src + (i64)(w + 2) * 2 * LL), v3 = cld(src + (i64)(w + 3) * 2 * LL);
            s += v0;
            s += v1;
            s += v2;
            s += v3;
          }
          for (; w < w1; ++w) s += cld(src + (i64)w * 2 * LL);
        }
        for (int off = 1; off < tpe; off <<= 1) s += __shfl_xor(s, off, 64);
        if (in && q == 0) cst(a.ddg + e, a.ninv * s);
      }
    }
    arrive();
    opaque();
    g_product(a.bgpub + (i64)parity * P * R * L, L, L, 3);
    if (!wait()) { status = 2; break; }

    // ---- chain ----
    opaque();
    T dreg[DPT];
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
      const int e = tid + kLoopThreads * q;
      dreg[q] = cld(a.ddg + (e < LL ? e : 0));
    }
    acc_t z[TPW], z2[TPW], z3[TPW];
    acc_t dg[TPW];
#pragma unroll
    for (int u = 0; u < TPW; ++u)
#pragma unroll
      for (int g = 0; g < 4; ++g)  // Dg(c, r): Dg = B^T M B / N is symmetric
        dg[u][g] = live[u] ? cld(a.ddg + LL + 16 * tn[u] + lr +
                                 (16 * tm[u] + SM<T>::row(lane, g)) * L)
                           : T(0);
    auto put_d = [&](T *dst) {
#pragma unroll
      for (int q = 0; q < DPT; ++q) {
        const int e = tid + kLoopThreads * q;
        if (e < LL) dst[e % L + (e / L) * LD] = dreg[q];
      }
    };
    put_d(s1);
    __syncthreads();
    // Z := Dg - D^T D
    mm(s1, s1, true, z);
#pragma unroll
    for (int u = 0; u < TPW; ++u) z[u] = dg[u] - z[u];
    put(s2, z);
    __syncthreads();
    mm(s2, s2, false, z2);
    put(s3, z2);
    rho = 4.0 * sqrt(sqrt(block_sum(norm2(z2))));  // 4 ||Z||_2 <= 4 ||Z^2||_F^(1/2)
    int t = 0;
    if (a.mode == 0)
      for (int q = kSeriesBlocks; q >= 1; --q)
        if (rho <= a.rho_max[q]) t = q;
    acc_t c[TPW], ci[TPW];
    if (t > 0) {
      mm(s2, s3, false, z3);
      const T *cf = coef + 4 * (t - 1), *cg = cf + kSeriesTerms;
#pragma unroll
      for (int u = 0; u < TPW; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          c[u][g] = block_at(cf, delta(u, g), z[u][g], z2[u][g], z3[u][g]);
          ci[u][g] = block_at(cg, delta(u, g), z[u][g], z2[u][g], z3[u][g]);
        }
      if (t > 1) {
        acc_t z4[TPW];
        mm(s3, s3, false, z4);
        __syncthreads();
        put(s1, z4);
        for (int i = t - 2; i >= 0; --i) {
          put(s2, c);
          put(s3, ci);
          __syncthreads();
          acc_t pc[TPW], pg[TPW];
          mm(s2, s1, false, pc);
          mm(s3, s1, false, pg);
          cf = coef + 4 * i;
          cg = cf + kSeriesTerms;
#pragma unroll
          for (int u = 0; u < TPW; ++u)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              c[u][g] = pc[u][g] + block_at(cf, delta(u, g), z[u][g], z2[u][g], z3[u][g]);
              ci[u][g] = pg[u][g] + block_at(cg, delta(u, g), z[u][g], z2[u][g], z3[u][g]);
            }
          __syncthreads();
        }
      } else {
        __syncthreads();
      }
    } else {
      // Newton-Schulz: rho = 4 ||Z^4||_F^(1/4); Y in s1, W in s2, E in s3
      acc_t z4[TPW];
      mm(s3, s3, false, z4);
      rho = 4.0 * sqrt(sqrt(sqrt(block_sum(norm2(z4)))));
      int k1 = 0, k2 = 0;
      if (!ns_counts<T>(rho, &k1, &k2)) { status = 1; break; }
      // c: Y, ci: W.  Stage 1 after its first step: Y1 = I - 2 Z - 8 Z2, W1 = I + 2 Z
#pragma unroll
      for (int u = 0; u < TPW; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          c[u][g] = delta(u, g) - T(2) * z[u][g] - T(8) * z2[u][g];
          ci[u][g] = delta(u, g) + T(2) * z[u][g];
        }
      auto step = [&] {  // E := 3I - W Y; Y := Y E / 2, W := E W / 2
        put(s1, c);
        put(s2, ci);
        __syncthreads();
        acc_t e[TPW], y[TPW], w[TPW];
        mm(s2, s1, false, e);
#pragma unroll
        for (int u = 0; u < TPW; ++u)
#pragma unroll
          for (int g = 0; g < 4; ++g) e[u][g] = T(3) * delta(u, g) - e[u][g];
        put(s3, e);
        __syncthreads();
        mm(s1, s3, false, y);
        mm(s3, s2, false, w);
#pragma unroll
        for (int u = 0; u < TPW; ++u) {
          c[u] = T(0.5) * y[u];
          ci[u] = T(0.5) * w[u];
        }
        __syncthreads();
      };
      for (int i = 1; i < k1; ++i) step();
      // stage 2 after its first step, P = Y: Y1 = (5 I + 4 P - P^2) / 8, W1 = (5 I - P) / 4
      put(s1, c);
      __syncthreads();
      acc_t pp[TPW];
      mm(s1, s1, false, pp);
#pragma unroll
      for (int u = 0; u < TPW; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          ci[u][g] = T(0.25) * (T(5) * delta(u, g) - c[u][g]);
          c[u][g] = T(0.625) * delta(u, g) + T(0.5) * c[u][g] - T(0.125) * pp[u][g];
        }
      __syncthreads();
      for (int i = 1; i < k2; ++i) step();
    }
    opaque();
    // ||C - I||_F over the l x l entries; F := C - D C^-1
    T sq = 0;
#pragma unroll
    for (int u = 0; u < TPW; ++u)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int r = 16 * tm[u] + SM<T>::row(lane, g), q = 16 * tn[u] + lr;
        const T d = c[u][g] - delta(u, g);
        if (live[u] && r < l && q < l) sq += d * d;
      }
    put_d(s1);
    put(s3, ci);
    err = sqrt(block_sum(sq));
    {
      acc_t f[TPW];
      mm(s1, s3, false, f);
#pragma unroll
      for (int u = 0; u < TPW; ++u) f[u] = c[u] - f[u];
      put(s2, f);
    }
    __syncthreads();

    // ---- X_+ := X F + (B / N) C^-1, B_+ := B F + Bg C^-1, Bg_+ := Bg F + G C^-1 (transposed) ----
    {
      opaque();
      constexpr int JOBS = 3 * NT, JPW = (JOBS + kLoopWaves - 1) / kLoopWaves;
      acc_t o[JPW];
#pragma unroll
      for (int u = 0; u < JPW; ++u) {
        const int job = wave + kLoopWaves * u;
        acc_t x = {0, 0, 0, 0}, y = {0, 0, 0, 0};
        if (job < JOBS) {
          const int j = job / NT, tc = job % NT;
          const T *pf = s2 + (16 * tc + lr) * LD + lk, *pc = s3 + (16 * tc + lr) * LD + lk;
          const T *px = st + (j * L + lk) * LDR + lr;
          const T *py = st + ((j + 1) * L + lk) * LDR + lr;
#pragma unroll 4
          for (int s = 0; s < 4 * NT; ++s) {
            x = SM<T>::mfma(pf[4 * s], px[4 * s * LDR], x);
            y = SM<T>::mfma(pc[4 * s], py[4 * s * LDR], y);
          }
          const T sc = j == 0 ? a.ninv : T(1);
#pragma unroll
          for (int g = 0; g < 4; ++g) x[g] += sc * y[g];
        }
        o[u] = x;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < JPW; ++u) {
        const int job = wave + kLoopWaves * u;
        if (job < JOBS) {
          const int j = job / NT, tc = job % NT;
#pragma unroll
          for (int g = 0; g < 4; ++g)
            st[(j * L + 16 * tc + SM<T>::row(lane, g)) * LDR + lr] = o[u][g];
        }
      }
      __syncthreads();
    }
    ++done;
    if (err <= a.tol || a.it0 + done == a.itmax) {
      status = 0;
      break;
    }
    opaque();
    gram();
    parity ^= 1;
    publish(parity);
  }
  __syncthreads();
  // the state: after the last iteration (0, 3), or the one that status 1 leaves to the caller
  for (int j = 0; j < (status == 1 ? 4 : status == 0 ? 1 : 3); ++j) save(j, a.state + (i64)j * Nl * l);
  if (blockIdx.x == 0 && tid == 0) {
    a.scal[0] = err;
    a.scal[1] = (double)(a.it0 + done);
    a.scal[2] = rho;
  }
  // one writer each, but for the word that every workgroup that timed out sets to the same value
  if (tid == 0 && blockIdx.x == 0) a.scal[3] = (double)status;
  if (tid == 0 && status == 2) a.scal[4] = 1.0;
}

template <typename T>
const double *series_rho_max() {
  static const struct Table {
    double v[kSeriesBlocks + 1];
    Table() {
      v[0] = 0;
      for (int t = 1; t <= kSeriesBlocks; ++t) {
        double lo = 0, hi = 0.5;  // series_blocks(0) = 1 <= t; at 0.5 it is 0
        for (int i = 0; i < 60; ++i) {
          const double mid = 0.5 * (lo + hi);
          const int b = series_blocks<T>(series_table<T>(), mid);
          if (b >= 1 && b <= t) lo = mid;
          else hi = mid;
        }
        v[t] = lo;
      }
    }
  } table;
  return table.v;
}

template <typename T, int NT>
void launch_loop(const KnLoopArgs<T> &a, int blocks) {
  using S = LoopLds<T, NT>;
  static_assert(S::bytes + 4096 <= 160 * 1024, "LDS budget");
  auto kern = kn_loop_kernel<T, NT>;
  HIP_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)S::bytes));
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kLoopThreads), S::bytes, ctx().stream, a);
  LAUNCH_CHECK();
}

}  // namespace

int kn_loop_mode() {
  const char *e = std::getenv("ISVD_KN_LOOP");
  return !e ? kKnLoopOn : e[0] == '0' ? kKnLoopOff : e[0] == '2' ? kKnLoopTimeout : kKnLoopOn;
}

template <typename T>
KnLoop<T>::KnLoop(i64 l_, i64 Nl_) : l(l_), Nl(Nl_) {
  ISVD_CHECK(kn_loop_fits((int)sizeof(T), l, Nl, ctx().cus), "kn_loop: l = %lld, Nl = %lld", l, Nl);
  blocks = (int)((Nl + kLoopRows - 1) / kLoopRows);
  const i64 L = (l + 15) / 16 * 16;
  buf.alloc(2 * (i64)blocks * kLoopRows * L + (i64)blocks * 2 * L * L + 2 * L * L);
  bar.alloc(2);
}

template <typename T>
void KnLoop<T>::run(const T *M, T ninv, T *state, bool resume, i64 it0, i64 itmax, i64 maxit,
                    double tol, int mode, double *scal) {
  const int nt = (int)((l + 15) / 16);
  const i64 L = 16 * nt;
  KnLoopArgs<T> a{};
  a.l = (int)l; a.Nl = (int)Nl; a.mode = mode; a.resume = resume ? 1 : 0;
  a.maxit = maxit; a.it0 = it0; a.itmax = itmax; a.tol = tol; a.ninv = ninv;
  a.spins = kn_loop_mode() == kKnLoopTimeout ? 0 : kChainSpinLimit;
  a.M = M; a.state = state; a.scal = scal; a.bar = bar.get();
  a.bgpub = buf.get();
  a.parts = a.bgpub + 2 * (i64)blocks * kLoopRows * L;
  a.ddg = a.parts + (i64)blocks * 2 * L * L;
  for (int i = 0; i < 2 * kSeriesTerms; ++i) a.coef[i] = series_table<T>()[i];
  for (int i = 0; i <= kSeriesBlocks; ++i) a.rho_max[i] = series_rho_max<T>()[i];
  zero_u64(bar.get(), 2);
  switch (nt) {
    case 1: launch_loop<T, 1>(a, blocks); break;
    case 2: launch_loop<T, 2>(a, blocks); break;
    case 3: launch_loop<T, 3>(a, blocks); break;
    case 4: launch_loop<T, 4>(a, blocks); break;
    default:
      if constexpr (sizeof(T) == 4) launch_loop<T, 5>(a, blocks);
      else fail("kn_loop: more than 64 FP64 columns do not fit in LDS");
  }
}

template struct KnLoop<double>;
template struct KnLoop<float>;

}  // namespace isvd
