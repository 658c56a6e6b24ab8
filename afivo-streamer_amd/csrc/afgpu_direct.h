// Exact solve on a uniformly refined level (mixed-precision form only).
//
// When every level up to lc covers the whole domain, the level-lc operator
// (afivo's constant-coefficient 3/5/7-point stencil with the physical
// boundary conditions folded in, m_af_stencil.f90:367-496,
// m_af_ghostcell.f90:173-279) is a Kronecker sum of 1-D operators, exactly
// like the level-1 box handled by k_coarse_solve.  The mixed-precision
// inner cycle solves its correction equation exactly on that level with the
// same fast diagonalisation, applied to the whole level at once: the
// level's boxes are gathered into one contiguous N^D grid (x fastest), each
// axis is transformed with the 1-D eigenvector matrix (small dense
// products, tiled through LDS), divided by the eigenvalue sums, and
// transformed back.  All transforms run in FP64.
#pragma once

#include <vector>

#include "afgpu_common.h"

namespace afg {

// Interior cells of the level's boxes <-> the contiguous grid.  `map` lists
// the box id of every box position (bx + nb*(by + nb*bz)), one workgroup
// per box; in a forest, run r's positions and grid follow those of run r-1.
template <int D, int NC, int BS, typename T>
__global__ void __launch_bounds__(BS) k_lc_gather(const int *__restrict__ map, int nb, const T *__restrict__ src,
                                                  double *__restrict__ A) {
  using G = Geo<D, NC>;
  const int b = blockIdx.x;
  const int id = map[b];
  if (id <= 0) return;  // run masked out
  const int per = (D == 3) ? nb * nb * nb : nb * nb;  // boxes of one run's level
  const int run = b / per, b0 = b % per;
  const int bx = b0 % nb, by = (b0 / nb) % nb, bz = (D == 3) ? b0 / (nb * nb) : 0;
  const int N = nb * NC;
  A += (size_t)run * ((D == 3) ? (size_t)N * N * N : (size_t)N * N);
  const T *u = src + (size_t)(id - 1) * Lay<D, NC, T>::STRIDE;
  for (int q = threadIdx.x; q < G::NINT; q += BS) {
    const int i = q % NC, j = (q / NC) % NC, k = (D == 3) ? q / (NC * NC) : 0;
    const size_t g = (size_t)(bx * NC + i) + (size_t)N * ((by * NC + j) + (size_t)N * (bz * NC + k));
    A[g] = (double)u[Lay<D, NC, T>::in_at(i + 1, j + 1, (D == 3) ? k + 1 : 0)];
  }
}

template <int D, int NC, int BS, typename T>
__global__ void __launch_bounds__(BS) k_lc_scatter(const int *__restrict__ map, int nb, const double *__restrict__ A,
                                                   T *__restrict__ dst) {
  using G = Geo<D, NC>;
  const int b = blockIdx.x;
  const int id = map[b];
  if (id <= 0) return;  // run masked out
  const int per = (D == 3) ? nb * nb * nb : nb * nb;
  const int run = b / per, b0 = b % per;
  const int bx = b0 % nb, by = (b0 / nb) % nb, bz = (D == 3) ? b0 / (nb * nb) : 0;
  const int N = nb * NC;
  A += (size_t)run * ((D == 3) ? (size_t)N * N * N : (size_t)N * N);
  T *u = dst + (size_t)(id - 1) * Lay<D, NC, T>::STRIDE;
  for (int q = threadIdx.x; q < G::NINT; q += BS) {
    const int i = q % NC, j = (q / NC) % NC, k = (D == 3) ? q / (NC * NC) : 0;
    const size_t g = (size_t)(bx * NC + i) + (size_t)N * ((by * NC + j) + (size_t)N * (bz * NC + k));
    u[Lay<D, NC, T>::in_at(i + 1, j + 1, (D == 3) ? k + 1 : 0)] = (T)A[g];
  }
}

// Transform along axis a >= 1 (y, or z in 3D):
//   out[.., i, .., x] = sum_m M[i][m] in[.., m, .., x]
// A workgroup takes TC consecutive x columns at one fixed value of the
// remaining coordinate; the N x TC input tile is staged in LDS, lanes run
// over the columns (coalesced) and the thread groups over output rows.
// With `div`, the result is divided by the eigenvalue sum of its cell
// (the last forward transform).
template <int D, int N>
__global__ void __launch_bounds__(256) k_lc_lines(const double *__restrict__ in, double *__restrict__ out,
                                                  const double *__restrict__ M, int axis, int div,
                                                  const double *__restrict__ eig, double lambda2) {
  constexpr int TC = (N < 64) ? N : (N == 64 ? 64 : 32);
  constexpr int G = 256 / TC;
  constexpr int RPT = (N + G - 1) / G;
  __shared__ double tile[N * TC];
  const int nxc = N / TC;
  const int xc = blockIdx.x % nxc, o = blockIdx.x / nxc;  // o: the other coordinate
  const int x0 = xc * TC;
  const size_t sa = (axis == 1) ? (size_t)N : (size_t)N * N;            // stride of the axis
  // stride of o (2D: the run of a forest)
  const size_t so = (D == 2) ? (size_t)N * N : ((axis == 1) ? (size_t)N * N : (size_t)N);
  const size_t base = (size_t)o * so + x0;
  for (int q = threadIdx.x; q < N * TC; q += 256) {
    const int m = q / TC, c = q % TC;
    tile[q] = in[base + (size_t)m * sa + c];
  }
  __syncthreads();
  const int c = threadIdx.x % TC, g = threadIdx.x / TC;
  double acc[RPT];
  for (int r = 0; r < RPT; r++) acc[r] = 0.0;
  for (int m = 0; m < N; m++) {
    const double t = tile[m * TC + c];
    for (int r = 0; r < RPT; r++) {
      const int i = g + r * G;
      if (i < N) acc[r] = acc[r] + M[i * N + m] * t;
    }
  }
  for (int r = 0; r < RPT; r++) {
    const int i = g + r * G;
    if (i >= N) break;
    double v = acc[r];
    if (div) {
      const int x = x0 + c;
      int y, z;
      if (D == 2) {
        y = i;
        z = 0;
      } else if (axis == 1) {
        y = i;
        z = o;
      } else {
        y = o;
        z = i;
      }
      double den = eig[x] + eig[N + y];
      if (D == 3) den = den + eig[2 * N + z];
      den = den - lambda2;
      v = v / den;
    }
    out[base + (size_t)i * sa + c] = v;
  }
}

// Transform along x (contiguous lines): out[r][i] = sum_m in[r][m] MT[m][i]
// with MT the transposed matrix.  A workgroup takes TR consecutive rows,
// staged in LDS (padded rows); lanes run over i (coalesced stores and
// matrix loads), thread groups over (i chunk, row subset).
template <int D, int N>
__global__ void __launch_bounds__(256) k_lc_rows(const double *__restrict__ in, double *__restrict__ out,
                                                 const double *__restrict__ MT, int nrows) {
  constexpr int TI = (N < 64) ? N : 64;
  constexpr int NIC = N / TI;
  constexpr int G = 256 / TI;
  constexpr int RG = G / NIC;
  constexpr int RPT = 16;
  constexpr int TR = RG * RPT;
  constexpr int LD = N + 1;
  __shared__ double tile[TR * LD];
  const int r0 = blockIdx.x * TR;
  for (int q = threadIdx.x; q < TR * N; q += 256) {
    const int rr = q / N, m = q % N;
    tile[rr * LD + m] = (r0 + rr < nrows) ? in[(size_t)(r0 + rr) * N + m] : 0.0;
  }
  __syncthreads();
  const int lane = threadIdx.x % TI, g = threadIdx.x / TI;
  const int ic = g % NIC, rg = g / NIC;
  const int i = ic * TI + lane;
  double acc[RPT];
  for (int r = 0; r < RPT; r++) acc[r] = 0.0;
  for (int m = 0; m < N; m++) {
    const double w = MT[m * N + i];
    for (int r = 0; r < RPT; r++) acc[r] = acc[r] + tile[(rg * RPT + r) * LD + m] * w;
  }
  for (int r = 0; r < RPT; r++) {
    const int row = r0 + rg * RPT + r;
    if (row < nrows) out[(size_t)row * N + i] = acc[r];
  }
}

// The same transforms for N = 64 and 128 as a tiled product (vector FMA)
//   out(i, col) = sum_m M[i][m] X(m, col)
// over 64 x 64 output tiles (i0.., col0..): chunks of 16 m are staged in LDS
// for both M and X (the next chunk is prefetched into registers while the
// current one is used), and each thread accumulates a 4 x 4 block.
// ROWS: X(m, col) = in[col*N + m] (the x transform, col = row of the grid);
// else X(m, col) = in[o*so + m*sa + x0 + col] (the y / z transforms).  With
// `div` (y/z forms only) the result is divided by the eigenvalue sum.
template <int D, int N, bool ROWS>
__global__ void __launch_bounds__(256) k_lc_gemm(const double *__restrict__ in, double *__restrict__ out,
                                                 const double *__restrict__ M, int axis, int div,
                                                 const double *__restrict__ eig, double lambda2) {
  static_assert(N == 64 || N == 128, "tiled transform for N = 64, 128");
  constexpr int T = 64, KC = 16, KP = KC + 1, NIT = N / T;
  __shared__ double Ms[T * KP];
  __shared__ double Xs[KC * T];
  const int it = blockIdx.x % NIT, rest = blockIdx.x / NIT;
  const int i0 = it * T;
  size_t sm, sc, base;
  int o = 0, x0 = 0;
  if (ROWS) {
    sm = 1;
    sc = N;
    base = (size_t)rest * T * N;
  } else {
    constexpr int nxc = N / T;
    const int xc = rest % nxc;
    o = rest / nxc;
    x0 = xc * T;
    sm = (axis == 1) ? (size_t)N : (size_t)N * N;
    const size_t so = (D == 2) ? (size_t)N * N : ((axis == 1) ? (size_t)N * N : (size_t)N);
    sc = 1;
    base = (size_t)o * so + x0;
  }
  const int tid = threadIdx.x;
  const int ti = ROWS ? (tid % 16) : (tid / 16);
  const int tc = ROWS ? (tid / 16) : (tid % 16);
  // global -> register staging of one chunk: 4 M and 4 X values per thread
  double pm[4], px[4];
  auto fetch = [&](int k0) {
    for (int u = 0; u < 4; u++) {
      const int q = tid + 256 * u;
      const int i = q / KC, kk = q % KC;
      pm[u] = M[(size_t)(i0 + i) * N + k0 + kk];
      int kx, c;
      if (ROWS) {
        kx = q % KC;
        c = q / KC;
      } else {
        c = q % T;
        kx = q / T;
      }
      px[u] = in[base + (size_t)(k0 + kx) * sm + (size_t)c * sc];
    }
  };
  auto stash = [&]() {
    for (int u = 0; u < 4; u++) {
      const int q = tid + 256 * u;
      Ms[(q / KC) * KP + q % KC] = pm[u];
      if (ROWS)
        Xs[(q % KC) * T + q / KC] = px[u];
      else
        Xs[(q / T) * T + q % T] = px[u];
    }
  };
  double acc[4][4];
  for (int r = 0; r < 4; r++)
    for (int q = 0; q < 4; q++) acc[r][q] = 0.0;
  fetch(0);
  for (int k0 = 0; k0 < N; k0 += KC) {
    stash();
    __syncthreads();
    if (k0 + KC < N) fetch(k0 + KC);
    for (int kk = 0; kk < KC; kk++) {
      double a[4], b[4];
      for (int r = 0; r < 4; r++) a[r] = Ms[(ti + 16 * r) * KP + kk];
      for (int q = 0; q < 4; q++) b[q] = Xs[kk * T + tc + 16 * q];
      for (int r = 0; r < 4; r++)
        for (int q = 0; q < 4; q++) acc[r][q] = acc[r][q] + a[r] * b[q];
    }
    __syncthreads();
  }
  for (int r = 0; r < 4; r++)
    for (int q = 0; q < 4; q++) {
      const int i = i0 + ti + 16 * r, c = tc + 16 * q;
      double v = acc[r][q];
      if (!ROWS && div) {
        const int x = x0 + c;
        int y, z;
        if (D == 2) {
          y = i;
          z = 0;
        } else if (axis == 1) {
          y = i;
          z = o;
        } else {
          y = o;
          z = i;
        }
        double den = eig[x] + eig[N + y];
        if (D == 3) den = den + eig[2 * N + z];
        den = den - lambda2;
        v = v / den;
      }
      out[base + (size_t)i * sm + (size_t)c * sc] = v;
    }
}

typedef double lc_double4 __attribute__((ext_vector_type(4)));
typedef float lc_float4 __attribute__((ext_vector_type(4)));

// Offset in the box pool (of values of type TS) of point (x, y, r) of the
// uniform level, stored as boxes of NC^D cells: r is z in 3D and the run of
// a forest in 2D; -1 when the box is masked out.
template <int D, int NC, typename TS>
__device__ inline long long lc_pool_offset(const int *__restrict__ map, int nb, int x, int y, int r) {
  using L = Lay<D, NC, TS>;
  int b, ck = 0;
  if (D == 3) {
    b = x / NC + nb * (y / NC + nb * (r / NC));
    ck = r % NC + 1;
  } else {
    b = x / NC + nb * (y / NC) + r * nb * nb;
  }
  const int id = map[b];
  return id > 0 ? (long long)(id - 1) * L::STRIDE + L::in_at(x % NC + 1, y % NC + 1, ck) : -1;
}

// The transforms on the FP64 matrix cores (v_mfma_f64_16x16x4f64, D = A B on
// 16 x 16 tiles, K = 4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and
// in register j D[4 j + l / 16][l % 16]).
//
// A workgroup of four or eight wavefronts takes C whole lines along the axis, so that
// everything it reads (the lines into LDS, its rows of the matrix into
// registers) is one round of independent loads with one barrier, and the
// last axis' forward transform, division and backward transform run on the
// lines while they are in LDS.  The passes are bound by that round and, on a
// 128^3 level, by the grid's traffic through the caches: 64 x 64 tiles
// in chunks of 32 along K took six passes and 98 us for 128^3 cells (now
// five and 71 us), 40 us for 64^3 (21), four passes and 36 us for one run of
// 128^2 (three, 18), 28 us for 13 runs of 64^2 (12).
//
// The matrices are packed in operand order (lc_pack): row tile by row tile,
// K step by K step, one value per lane.
//
// FOLD (an axis whose 1-D operator is symmetric under reversal,
// m -> N - 1 - m, N = 128): its eigenvectors are even or odd, so a transform
// needs half the products.  Forward: the even modes (rows 0..N/2 - 1 of the
// matrix, N x N/2) take u_m + u_{N-1-m}, the odd ones u_m - u_{N-1-m}, over
// K = N/2.  Backward: the matrix (N/2 x N) gives the sums over the even modes
// (E) and the odd ones (O), u_m = E + O and u_{N-1-m} = E - O.
inline std::vector<double> lc_pack(const double *M, int rows, int cols) {
  std::vector<double> p((size_t)rows * cols);
  size_t o = 0;
  for (int rt = 0; rt < rows / 16; rt++)
    for (int st = 0; st < cols / 4; st++)
      for (int l = 0; l < 64; l++) p[o++] = M[(size_t)(rt * 16 + l % 16) * cols + 4 * st + l / 16];
  return p;
}
template <int N, bool FOLD>
struct LcGeo {
  static constexpr int W = (N == 128 && !FOLD) ? 8 : 4;  // wavefronts of a workgroup
  static constexpr int NWR = (N / 16 < W) ? N / 16 : W;  // of them along the output index
  static constexpr int NWC = W / NWR;                    // and along the lines
  static constexpr int C = 16 * NWC;                     // lines per workgroup
  static constexpr int RT = N / 16 / NWR;                // 16-row tiles per wavefront
  static constexpr int BT = 64 * W;
};
// A packed 16-row matrix tile over ST steps of K, one value per lane and
// step in registers: loaded ahead of the barrier that the lines wait for.
template <int ST>
struct LcTile {
  double m[ST];
  __device__ void load(const double *__restrict__ mp) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int st = 0; st < ST; st++) m[st] = mp[st * 64 + lane];
  }
};
// One product of a wavefront over steps S0 .. S0 + ST - 1 of the tile, the
// other operand from LDS, at step s at xs[s * step].
template <int S0, int ST, bool ROWS, int TST>
__device__ inline lc_double4 lc_product(const LcTile<TST> &mt, const double *xs, int step) {
  lc_double4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int st = 0; st < ST; st++) {
    const double x = xs[st * step];
    acc = ROWS ? __builtin_amdgcn_mfma_f64_16x16x4f64(x, mt.m[S0 + st], acc, 0, 0, 0)
               : __builtin_amdgcn_mfma_f64_16x16x4f64(mt.m[S0 + st], x, acc, 0, 0, 0);
  }
  return acc;
}

// The x transforms: IO 1 forward, the rows read from the box pool `pin`;
// IO 2 backward, the result written to the box pool `pout`.
template <int D, int N, int IO, int NC, typename TS, bool FOLD>
__global__ void __launch_bounds__((LcGeo<N, FOLD>::BT), 4) k_lc_x(const double *__restrict__ in, double *__restrict__ out,
                                              const double *__restrict__ M, const int *__restrict__ map, int nb,
                                              const TS *__restrict__ pin, TS *__restrict__ pout) {
  using LG = LcGeo<N, FOLD>;
  constexpr int C = LG::C, S = N + 4;  // (row stride: 16 rows and 4 steps of K over all LDS banks)
  constexpr int H = N / 2, PER = C * N / LG::BT;
  __shared__ double xs[C * S];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wr = w % LG::NWR, wc = w / LG::NWR;
  const int r0 = blockIdx.x * C;  // first grid row
  // a wavefront's row tiles (folded backward: one tile over E and O)
  constexpr int RT = (IO == 2 && FOLD) ? 1 : LG::RT, KS = (IO == 1 && FOLD ? H : N) / 4;
  constexpr int EARLY = (KS * RT <= 32) ? RT : 1;  // (tiles held in registers from the start)
  const double *mw = M + (size_t)wr * RT * KS * 64;
  LcTile<KS> mt[EARLY];
  // The rows lie on one plane z (or in one run), in the boxes yb = 0 ..
  // C / NC - 1 from the first row's on: where column x begins in box yb
  // (negative: masked out), and cell (x, row) from there on.
  using L = Lay<D, NC, TS>;
  const int z = r0 / N, y0 = r0 % N, kz = (D == 3) ? z % NC + 1 : 0;
  auto box_at = [&](int x, int yb) {
    const int b = x / NC + nb * (y0 / NC + yb) + ((D == 3) ? nb * nb * (z / NC) : nb * nb * z);
    const int id = map[b];
    return id > 0 ? (long long)(id - 1) * L::STRIDE : -1ll;
  };
  auto in_box = [&](int x, int r) { return L::in_at(x % NC + 1, r % NC + 1, kz); };
  if constexpr (IO == 1) {
    // RU rows per step of the loads: the box of a step's rows is known
    constexpr int RU = LG::BT / (FOLD ? H : N), YB = C / NC;
    static_assert(RU <= NC && NC % RU == 0 && C % NC == 0, "a step's rows lie in one box");
    const int xa = tid % (FOLD ? H : N);
    long long ba[YB], bb[YB];
#pragma unroll
    for (int yb = 0; yb < YB; yb++) {
      ba[yb] = box_at(xa, yb);
      if (FOLD) bb[yb] = box_at(N - 1 - xa, yb);
    }
    auto val = [&](long long base, int x, int r) { return base >= 0 ? (double)pin[base + in_box(x, r)] : 0.0; };
    if constexpr (FOLD) {
      double a[PER / 2], b[PER / 2];
#pragma unroll
      for (int u = 0; u < PER / 2; u++) {
        const int r = (tid + u * LG::BT) / H;
        a[u] = val(ba[u * RU / NC], xa, r);
        b[u] = val(bb[u * RU / NC], N - 1 - xa, r);
      }
      for (int t = 0; t < EARLY; t++) mt[t].load(mw + (size_t)t * KS * 64);
#pragma unroll
      for (int u = 0; u < PER / 2; u++) {
        const int q = tid + u * LG::BT, x = q % H, r = q / H;
        xs[r * S + x] = a[u] + b[u];
        xs[r * S + H + x] = a[u] - b[u];
      }
    } else {
      double a[PER];
#pragma unroll
      for (int u = 0; u < PER; u++) {
        a[u] = val(ba[u * RU / NC], xa, (tid + u * LG::BT) / N);
      }
      for (int t = 0; t < EARLY; t++) mt[t].load(mw + (size_t)t * KS * 64);
#pragma unroll
      for (int u = 0; u < PER; u++) {
        const int q = tid + u * LG::BT;
        xs[(q / N) * S + q % N] = a[u];
      }
    }
  } else {
    double a[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) a[u] = in[(size_t)r0 * N + tid + u * LG::BT];
    for (int t = 0; t < EARLY; t++) mt[t].load(mw + (size_t)t * KS * 64);
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int q = tid + u * LG::BT;
      xs[(q / N) * S + q % N] = a[u];
    }
  }
  __syncthreads();
  const double *x0 = xs + (16 * wc + (lane & 15)) * S + (lane >> 4);
  if constexpr (IO == 2 && FOLD) {
    // output tile m = 16 wr .. of the first half, and its mirror
    const lc_double4 E = lc_product<0, H / 4, true>(mt[0], x0, 4);
    const lc_double4 O = lc_product<H / 4, H / 4, true>(mt[0], x0 + H, 4);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int r = 16 * wc + 4 * j + (lane >> 4), m = 16 * wr + (lane & 15), yb = (16 * wc + 4 * j) / NC;
      const long long lo = box_at(m, yb), hi = box_at(N - 1 - m, yb);
      if (lo >= 0) pout[lo + in_box(m, r)] = (TS)(E[j] + O[j]);
      if (hi >= 0) pout[hi + in_box(N - 1 - m, r)] = (TS)(E[j] - O[j]);
    }
  } else {
#pragma unroll
    for (int t = 0; t < RT; t++) {
      const int rt = wr * RT + t;  // (folded: the first half of the row tiles are the even modes)
      const double *xt = x0 + (FOLD && rt >= N / 32 ? H : 0);
      if (t >= EARLY) mt[0].load(mw + (size_t)t * KS * 64);
      const lc_double4 v = lc_product<0, KS, true>(mt[t < EARLY ? t : 0], xt, 4);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int r = 16 * wc + 4 * j + (lane >> 4), m = 16 * rt + (lane & 15);
        if constexpr (IO == 2) {
          const long long base = box_at(m, (16 * wc + 4 * j) / NC);
          if (base >= 0) pout[base + in_box(m, r)] = (TS)v[j];
        } else {
          out[(size_t)(r0 + r) * N + m] = v[j];
        }
      }
    }
  }
}

// The transforms along y and z: DIR 1 forward (Mf), 2 backward (Mb), 3 the
// last axis: forward, division by the eigenvalue sums and backward.  A
// workgroup takes C neighbouring columns x at one value o of the remaining
// coordinate (z for the y axis, y for the z axis; the run in 2D).  The last
// axis is done in place (in == out): a workgroup reads and writes the same
// lines, all of them into LDS before a barrier and none stored before it.
template <int D, int N, int DIR, bool FOLD>
__global__ void __launch_bounds__((LcGeo<N, FOLD>::BT), 4) k_lc_line(const double *in, double *out,
                                                 const double *__restrict__ Mf, const double *__restrict__ Mb, int axis,
                                                 const double *__restrict__ eig, double lambda2) {
  using LG = LcGeo<N, FOLD>;
  constexpr int C = LG::C, H = N / 2, PER = C * N / LG::BT, NXC = N / C;
  __shared__ double xs[N * C];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wr = w % LG::NWR, wc = w / LG::NWR;
  const int x0 = (blockIdx.x % NXC) * C, o = blockIdx.x / NXC;
  const size_t sm = (axis == 1) ? (size_t)N : (size_t)N * N;
  const size_t so = (D == 2) ? (size_t)N * N : ((axis == 1) ? (size_t)N * N : (size_t)N);
  const size_t base = (size_t)o * so + x0;
  // a wavefront's row tiles, forward and (folded: one tile over E and O) backward
  constexpr int RT = LG::RT, KS = (FOLD ? H : N) / 4, RB = FOLD ? 1 : RT, KB = N / 4;
  constexpr int EF = (KS * RT <= 32) ? RT : 1, EB = (KB * RB <= 32) ? RB : 1;  // (tiles held from the start)
  const double *mfw = Mf + (size_t)wr * RT * KS * 64, *mbw = Mb + (size_t)wr * RB * KB * 64;
  LcTile<KS> mf[EF];
  LcTile<KB> mb[EB];
  auto early = [&] {
    if constexpr (DIR & 1)
      for (int t = 0; t < EF; t++) mf[t].load(mfw + (size_t)t * KS * 64);
    else
      for (int t = 0; t < EB; t++) mb[t].load(mbw + (size_t)t * KB * 64);
  };
  if constexpr (FOLD && (DIR & 1)) {
    double a[PER / 2], b[PER / 2];
#pragma unroll
    for (int u = 0; u < PER / 2; u++) {
      const int q = tid + u * LG::BT, k = q / C, c = q % C;
      a[u] = in[base + (size_t)k * sm + c];
      b[u] = in[base + (size_t)(N - 1 - k) * sm + c];
    }
    early();
#pragma unroll
    for (int u = 0; u < PER / 2; u++) {
      const int q = tid + u * LG::BT;
      xs[q] = a[u] + b[u];
      xs[H * C + q] = a[u] - b[u];
    }
  } else {
    double a[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int q = tid + u * LG::BT;
      a[u] = in[base + (size_t)(q / C) * sm + q % C];
    }
    early();
#pragma unroll
    for (int u = 0; u < PER; u++) xs[tid + u * LG::BT] = a[u];
  }
  __syncthreads();
  const int col = 16 * wc + (lane & 15);
  const double *b0 = xs + (lane >> 4) * C + col;
  if constexpr (DIR & 1) {
    lc_double4 v[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) {
      if (t >= EF) mf[0].load(mfw + (size_t)t * KS * 64);
      v[t] = lc_product<0, KS, false>(mf[t < EF ? t : 0], b0 + (FOLD && wr * RT + t >= N / 32 ? H * C : 0), 4 * C);
    }
    if constexpr (DIR == 3) {
      for (int t = 0; t < EB; t++) mb[t].load(mbw + (size_t)t * KB * 64);
      __syncthreads();  // (every wavefront is done with the lines)
    }
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int p = 16 * (wr * RT + t) + 4 * j + (lane >> 4);
        if constexpr (DIR == 3) {
          double den = eig[x0 + col] + eig[N + ((D == 3) ? o : p)];
          if (D == 3) den = den + eig[2 * N + p];
          den = den - lambda2;
          xs[p * C + col] = v[t][j] / den;
        } else {
          out[base + (size_t)p * sm + col] = v[t][j];
        }
      }
    if constexpr (DIR == 1) return;
    __syncthreads();
  }
  if constexpr (DIR & 2) {
    if constexpr (FOLD) {
      const lc_double4 E = lc_product<0, H / 4, false>(mb[0], b0, 4 * C);
      const lc_double4 O = lc_product<H / 4, H / 4, false>(mb[0], b0 + H * C, 4 * C);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int p = 16 * wr + 4 * j + (lane >> 4);
        out[base + (size_t)p * sm + col] = E[j] + O[j];
        out[base + (size_t)(N - 1 - p) * sm + col] = E[j] - O[j];
      }
    } else {
#pragma unroll
      for (int t = 0; t < RB; t++) {
        if (t >= EB) mb[0].load(mbw + (size_t)t * KB * 64);
        const lc_double4 v = lc_product<0, KB, false>(mb[t < EB ? t : 0], b0, 4 * C);
#pragma unroll
        for (int j = 0; j < 4; j++) out[base + (size_t)(16 * (wr * RB + t) + 4 * j + (lane >> 4)) * sm + col] = v[j];
      }
    }
  }
}

// The transforms in single precision (the mixed form's inner cycle, option
// AFGPU_OPT_DIRECT_F32), 64 x 64 output tiles in chunks of 32 along K: grids,
// matrices and eigenvalues in FP32, products on the FP32 matrix cores
// (v_mfma_f32_16x16x4f32: the operands as in the FP64 form, result register
// j of lane l holding row 4 (l / 16) + j, column l % 16 of the 16 x 16
// block).  ROWS: D[p][q], p = grid row, q = output index (IO 1: the rows read
// from the box pool, 2: written to it); else p = output index, q = column x.
template <int D, int N, bool ROWS, int IO = 0, int NC = 16>
__global__ void __launch_bounds__(256) k_lc_mfma32(const float *__restrict__ in, float *__restrict__ out,
                                                   const float *__restrict__ M, int axis, int div,
                                                   const float *__restrict__ eig, float lambda2,
                                                   const int *__restrict__ map, int nb, const float *__restrict__ pin,
                                                   float *__restrict__ pout) {
  static_assert(IO == 0 || ROWS, "box-pool input and output in the x form only");
  static_assert(N == 64 || N == 128, "matrix-core transform for N = 64, 128");
  constexpr int T = 64, KC = 32, AP = KC + 1, BP = T + 1, NT = N / T;
  constexpr int PER = T * KC / 256;  // values of each operand tile per thread
  __shared__ float As[T * AP];   // As[p][kk]
  __shared__ float Bs[KC * BP];  // Bs[kk][q]
  // blocks: ROWS: (output tiles) x (row tiles); else (output tiles) x
  // (column tiles) x (the remaining coordinate)
  const int t0 = blockIdx.x % NT, rest = blockIdx.x / NT;
  size_t sm = 1, base = 0;
  int o = 0, x0 = 0, p0 = 0, q0 = 0;
  if (ROWS) {
    p0 = rest * T;  // grid rows
    q0 = t0 * T;    // output index i
  } else {
    p0 = t0 * T;  // output index i
    x0 = (rest % NT) * T;
    o = rest / NT;
    q0 = 0;
    sm = (axis == 1) ? (size_t)N : (size_t)N * N;
    const size_t so = (D == 2) ? (size_t)N * N : ((axis == 1) ? (size_t)N * N : (size_t)N);
    base = (size_t)o * so + x0;
  }
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wp = (w >> 1) * 32, wq = (w & 1) * 32;
  // one K chunk of both operands, global -> registers (consecutive threads
  // take consecutive addresses) and registers -> LDS
  float pa[PER], pb[PER];
  auto fetch = [&](int k0) {
    for (int u = 0; u < PER; u++) {
      const int q = tid + 256 * u;
      const int pp = q / KC, kk = q % KC;
      if (IO == 1) {
        const int row = p0 + pp;
        const long long off = lc_pool_offset<D, NC, float>(map, nb, k0 + kk, row % N, row / N);
        pa[u] = off >= 0 ? pin[off] : 0.0f;
      } else {
        pa[u] = ROWS ? in[(size_t)(p0 + pp) * N + k0 + kk] : M[(size_t)(p0 + pp) * N + k0 + kk];
      }
      if (ROWS) {
        pb[u] = M[(size_t)(q0 + pp) * N + k0 + kk];
      } else {
        const int kb = q / T, qq = q % T;
        pb[u] = in[base + (size_t)(k0 + kb) * sm + qq];
      }
    }
  };
  auto stash = [&]() {
    for (int u = 0; u < PER; u++) {
      const int q = tid + 256 * u;
      As[(q / KC) * AP + q % KC] = pa[u];
      if (ROWS)
        Bs[(q % KC) * BP + q / KC] = pb[u];
      else
        Bs[(q / T) * BP + q % T] = pb[u];
    }
  };
  lc_float4 acc[2][2];
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++) acc[a][b] = lc_float4{0.0f, 0.0f, 0.0f, 0.0f};
  fetch(0);
  for (int k0 = 0; k0 < N; k0 += KC) {
    stash();
    __syncthreads();
    if (k0 + KC < N) fetch(k0 + KC);
    for (int ks = 0; ks < KC; ks += 4) {
      const int kk = ks + (lane >> 4);
      float a[2], b[2];
      for (int t = 0; t < 2; t++) {
        a[t] = As[(wp + 16 * t + (lane & 15)) * AP + kk];
        b[t] = Bs[kk * BP + wq + 16 * t + (lane & 15)];
      }
      for (int ta = 0; ta < 2; ta++)
        for (int tb = 0; tb < 2; tb++)
          acc[ta][tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[ta], b[tb], acc[ta][tb], 0, 0, 0);
    }
    __syncthreads();
  }
  for (int ta = 0; ta < 2; ta++)
    for (int tb = 0; tb < 2; tb++)
      for (int j = 0; j < 4; j++) {
        const int pp = p0 + wp + 16 * ta + 4 * (lane >> 4) + j;
        const int qq = q0 + wq + 16 * tb + (lane & 15);
        float v = acc[ta][tb][j];
        if (ROWS && IO == 2) {
          const long long off = lc_pool_offset<D, NC, float>(map, nb, qq, pp % N, pp / N);
          if (off >= 0) pout[off] = v;
        } else if (ROWS) {
          out[(size_t)pp * N + qq] = v;
        } else {
          if (div) {
            const int x = x0 + qq;
            int y, z;
            if (D == 2) {
              y = pp;
              z = 0;
            } else if (axis == 1) {
              y = pp;
              z = o;
            } else {
              y = o;
              z = pp;
            }
            float den = eig[x] + eig[N + y];
            if (D == 3) den = den + eig[2 * N + z];
            den = den - lambda2;
            v = v / den;
          }
          out[base + (size_t)pp * sm + qq] = v;
        }
      }
}

}  // namespace afg
