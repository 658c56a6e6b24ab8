// The coarse levels of the FP64 multigrid in one workgroup per run.
//
// The lowest levels of a tree have few boxes (a quarter or an eighth of the
// level above), so a V-cycle's kernels there do almost nothing: on MI355X a
// dependent launch in a captured graph costs 1.6 us before it does any work
// and its chain of dependent loads (list -> box record -> neighbour -> cell)
// 1.5 us more, and the 18 launches a level takes cost the same on level 2 as
// on level 7.  Here one workgroup holds phi of all boxes of levels 1..lt of
// its run in LDS and works through the host's list of operations (half-sweeps,
// ghost fills, restriction, coarse right-hand sides, the level-1 solve,
// prolongation, residuals), with a barrier between two operations instead of
// a launch.  The expressions, their operands and their order are those of the
// level kernels (afgpu_mg.h), so the results are identical; the neighbours of
// a box follow from its position, the levels being uniformly refined.
//
// Bound by the length of that list: a barrier and the instructions of a
// phase, 0.3 to 1 us each with one workgroup's 16 waves, so indices and
// coefficients come from tables filled once per launch.  Measured: a V-cycle
// on four levels of 8^2 boxes (64^2 cells) 45 us, of which 4 us load and
// store the levels, against 165 us for its 55 launches; the level-1 solve of
// a 16^3 box 17 us (52 us with its matrices read from memory).
#pragma once

#include <type_traits>

#include "afgpu_mg.h"

namespace afg {

enum TailOpCode {
  TL_SWEEP = 0,  // a: half-sweeps, b: TailSweep flags
  TL_GC,         // a: edges and corners too
  TL_RESTRICT,   // level -> level - 1; a: keep the residual in tmp
  TL_RHS,        // on the parents of the level; a: tmp = phi
  TL_SOLVE,      // level 1
  TL_COPY,       // tmp = phi
  TL_SUB,        // tmp = phi - tmp on the parents of the level
  TL_PROLONG,    // phi of the level += P(tmp of level - 1)
  TL_RESID,      // tmp = rhs - L phi, max over leaves into red
  TL_RESET       // red = 0
};
// The first half-sweep reads the stored ghost layer; after the last one the
// ghost layer is filled, with edges and corners.
enum TailSweep { TS_STORED = 1, TS_GC = 2, TS_CORNERS = 4 };
struct TailOp {
  unsigned char op, lvl, a, b;
};
constexpr int TAIL_MAX_OPS = 240;
constexpr int TAIL_NT = 1024;
// Levels held: 4096 cells on the finest one (two cells of a colour per
// thread): 85 boxes of 8^2, 21 of 16^2, 9 of 8^3 or one of 16^3.  phi of all
// of them and rhs and tmp of the levels below the finest are in LDS (99, 78,
// 86 and 46 KB, with the tables and the level-1 matrices 120, 100, 111 and
// 98); rhs and tmp of the finest, which a cycle touches a few times only, stay
// in memory.
template <int D, int NC>
struct TailGeo {
  static constexpr int LT = (D == 2) ? (NC == 8 ? 4 : 3) : (NC == 8 ? 2 : 1);
  static constexpr int off(int lvl) {  // slots of the levels below
    int n = 0;
    for (int l = 1; l < lvl; l++) n += 1 << (D * (l - 1));
    return n;
  }
  static constexpr int SLOTS = off(LT + 1);
  static constexpr int LOW = off(LT);  // slots with rhs and tmp in LDS
  // Index tables, the same for every run: a word per face ghost, in the
  // order box, colour of the cell behind it, face, position, and a word per
  // edge and corner cell.  Cells are numbered over the slots (below 2^14).
  static constexpr int NGB = D * Geo<D, NC>::NTAN;  // ghosts of a box next to one colour
  static constexpr int NX = (D == 3 ? 12 * NC : 0) + (1 << D);
  static constexpr int N_GH = SLOTS * 2 * NGB, N_CR = SLOTS * NX;
  static constexpr int COLS = NC * ((1 << LT) - 1);  // cell columns along x of all levels
  // k_tail's LDS arrays
  static constexpr int N_PHI = SLOTS * Geo<D, NC>::NCELL;
  static constexpr int N_LOW = LOW ? LOW * Geo<D, NC>::NCELL : 2;  // (2: a word that nothing reads)
  static constexpr int N_MAT = 2 * D * NC * (NC + 1);
  static constexpr int N_CYL = D == 2 ? COLS : 1;
  static constexpr int N_F64 =
      N_PHI + 2 * N_LOW + Geo<D, NC>::NINT + N_MAT + D * NC + LT * (8 + 4 * D) + N_CYL * 5;
  static constexpr int LDS = 8 * N_F64 + 4 * (N_GH + N_CR + 2 * SLOTS);
  static_assert(LDS <= 160 * 1024, "the LDS of a CU");
};
// A face ghost: bits 0-13 its cell, 14-27 the cell it is formed from (the
// neighbour's, or the box's first one; the second one lies as far again),
// 28-31 TG_COPY or the physical face.
constexpr unsigned TG_COPY = 15;
// An edge or corner cell: bits 0-13 the cell, 14-27 the diagonal neighbour's
// (bit 31 set) or bits 14-19 the direction codes (two bits an axis: 0 along
// the edge, 1 low, 2 high).
template <int D, int NC>
inline void tail_tables(unsigned *gh, unsigned *cr) {
  using G = Geo<D, NC>;
  using TG = TailGeo<D, NC>;
  static_assert(TG::SLOTS * G::NCELL < (1 << 14), "cells numbered in 14 bits");
  for (int l = 1; l <= TG::LT; l++) {
    const int n1 = 1 << (l - 1), n_box = 1 << (D * (l - 1));
    for (int p = 0; p < n_box; p++) {
      const int x[3] = {p % n1, (p / n1) % n1, p / (n1 * n1)}, slot = TG::off(l) + p;
      const int step[3] = {1, n1, n1 * n1};
      for (int c = 0; c < 2; c++)
        for (int e = 0; e < TG::NGB; e++) {
          constexpr int NE = G::NTAN / 2;
          const int nb = e / NE, r = e % NE, d = nb / 2, low = (nb & 1) == 0;
          const int b = (D == 3) ? r / (NC / 2) + 1 : 0;
          const int a = 2 * (r % (NC / 2)) + 1 + ((c + (low ? 1 : NC) + b + 1) & 1);
          auto cell = [&](int pn) {
            const int i = (d == 0) ? pn : a, j = (d == 1) ? pn : (D == 2 || d == 0) ? a : b;
            return G::idx(i, j, (D == 2) ? 0 : (d == 2) ? pn : b);
          };
          const bool inside = low ? x[d] > 0 : x[d] < n1 - 1;
          const unsigned dst = slot * G::NCELL + cell(low ? 0 : NC + 1);
          const unsigned src = inside ? (slot + (low ? -step[d] : step[d])) * G::NCELL + cell(low ? NC : 1)
                                      : slot * G::NCELL + cell(low ? 1 : NC);
          gh[(slot * 2 + c) * TG::NGB + e] = dst | src << 14 | (inside ? TG_COPY : (unsigned)nb) << 28;
        }
      for (int e = 0; e < TG::NX; e++) {
        constexpr int NED = (D == 3) ? 12 * NC : 0;
        const bool edge = e < NED;
        const int n = edge ? e / NC : e - NED, dim = edge ? n >> 2 : -1;
        int dir[3] = {0, 0, 0}, lo[3] = {0, 0, 0}, bit = 0, pn = slot;
        bool inside = true;
        for (int d = 0; d < D; d++) {
          if (d == dim) {
            lo[d] = e % NC + 1;
            continue;
          }
          dir[d] = 2 * ((n >> bit++) & 1) - 1;
          lo[d] = dir[d] > 0 ? NC + 1 : 0;
          inside = inside && x[d] + dir[d] >= 0 && x[d] + dir[d] < n1;
          pn += dir[d] * step[d];
        }
        unsigned w = slot * G::NCELL + G::idx(lo[0], lo[1], lo[2]);
        if (inside)
          w |= 1u << 31 | (unsigned)(pn * G::NCELL + G::idx(lo[0] - dir[0] * NC, lo[1] - dir[1] * NC, lo[2] - dir[2] * NC))
                              << 14;
        else
          for (int d = 0; d < D; d++) w |= (dir[d] == 0 ? 0u : dir[d] < 0 ? 1u : 2u) << (14 + 2 * d);
        cr[slot * TG::NX + e] = w;
      }
    }
  }
}
struct TailArgs {
  int *map;  // box id of every slot, [run][SLOTS]: levels in turn, x fastest; negated: run masked out
  const unsigned *gh, *cr;  // tail_tables
  const DBox *boxes;
  double *phi, *rhs, *tmp;
  VarBc m;
  double lambda2;
  const double *vinv, *v, *eig;
  unsigned long long *red;
  int cyl, lt, n_ops;
  TailOp ops[TAIL_MAX_OPS];
};

template <int D, int NC>
__global__ void __launch_bounds__(TAIL_NT) k_tail(TailArgs A) {
  using G = Geo<D, NC>;
  using TG = TailGeo<D, NC>;
  constexpr int HALF = G::NINT / 2, NCELL = G::NCELL;
  constexpr int H = NC / 2, NQ = G::NINT >> D, NCH = 1 << D, NMAT = TG::N_MAT;
  constexpr int TOP = 1 << (D * (TG::LT - 1));  // boxes of the finest level
  constexpr int PER = (TOP * HALF + TAIL_NT - 1) / TAIL_NT;
  constexpr int NGB = TG::NGB, NX = TG::NX;
  constexpr int GPER = (TOP * NGB + TAIL_NT - 1) / TAIL_NT;
  __shared__ __align__(16) double s_phi[TG::N_PHI];
  __shared__ __align__(16) double s_rhs[TG::N_LOW], s_tmp[TG::N_LOW];
  __shared__ double s_buf[G::NINT];            // level-1 solve
  __shared__ double s_mat[NMAT + D * NC];      // its matrices, padded rows, and eigenvalues
  __shared__ double s_st[TG::LT][8];           // the levels' stencils, and 1 / the diagonal
  __shared__ double s_bc[TG::LT][2 * D][2];    // phys_coeffs of their faces
  __shared__ double s_cyl[TG::N_CYL][5];       // per column: c1, c2, c3, 1 / c1, restriction weight
  __shared__ unsigned s_gh[TG::N_GH], s_cr[TG::N_CR];
  __shared__ int s_id[TG::SLOTS];
  __shared__ int s_par[TG::SLOTS];
  const int tid = threadIdx.x, run = blockIdx.x;
  const int *map = A.map + (size_t)run * TG::SLOTS;
  if (map[0] <= 0) return;  // run masked out
  auto level_off = [](int lvl) { return ((1 << (D * (lvl - 1))) - 1) / (NCH - 1); };
  const int n_slots = level_off(A.lt + 1), n_low = min(n_slots, TG::LOW);
  typedef double d2 __attribute__((ext_vector_type(2)));
  constexpr int NV = NCELL / 2;
  static_assert(NCELL % 2 == 0, "boxes of whole 16-byte words");
  for (int q = tid; q < 2 * D * NC * NC; q += TAIL_NT)
    s_mat[(q / NC) * (NC + 1) + q % NC] = (q < D * NC * NC) ? A.vinv[q] : A.v[q - D * NC * NC];
  for (int q = tid; q < D * NC; q += TAIL_NT) s_mat[NMAT + q] = A.eig[q];
  for (int q = tid; q < n_slots; q += TAIL_NT) {
    const int id = map[q];
    const DBox &bx = A.boxes[id - 1];
    s_id[q] = id;
    s_par[q] = bx.children[0] > 0;
  }
  for (int q = tid; q < n_slots * 2 * NGB; q += TAIL_NT) s_gh[q] = A.gh[q];
  for (int q = tid; q < n_slots * NX; q += TAIL_NT) s_cr[q] = A.cr[q];
  const double run_val = A.m.run_val ? A.m.run_val[run] : 0.0;
  const bool cyl = A.cyl != 0;
  if (tid < A.lt) {
    const DBox &bx = A.boxes[map[level_off(tid + 1)] - 1];
    const Sten<D, double> st = lpl_stencil<D, double>(bx, A.lambda2);
    for (int q = 0; q <= 2 * D; q++) s_st[tid][q] = st.c[q];
    s_st[tid][7] = 1.0 / st.c[0];
    for (int nb = 0; nb < 2 * D; nb++) phys_coeffs<D, double>(bx.dr, A.m, run_val, nb, s_bc[tid][nb][0], s_bc[tid][nb][1]);
  }
  if (D == 2 && cyl) {
    // column i of the box at x of level l (the boxes above it have the
    // same r_min)
    for (int q = tid; q < NC * ((1 << A.lt) - 1); q += TAIL_NT) {
      const int l = 32 - __clz(q / NC + 1), x = q / NC + 1 - (1 << (l - 1)), i = q % NC + 1;
      const DBox &bx = A.boxes[map[level_off(l) + x] - 1];
      const Sten<D, double> st = lpl_stencil<D, double>(bx, A.lambda2);
      double c1, c2, c3;
      cyl_coeffs<double>(bx, i, st.c, c1, c2, c3);
      s_cyl[q][0] = c1;
      s_cyl[q][1] = c2;
      s_cyl[q][2] = c3;
      s_cyl[q][3] = 1.0 / c1;
      s_cyl[q][4] = restrict_weight<double>(bx, i);
    }
  }
  for (int q = tid; q < n_slots * NV; q += TAIL_NT) {
    const int s = q / NV, x = q - s * NV;
    const size_t base = (size_t)(map[s] - 1) * NCELL;
    reinterpret_cast<d2 *>(s_phi)[q] = reinterpret_cast<const d2 *>(A.phi + base)[x];
    if (TG::LOW && s < n_low) {
      reinterpret_cast<d2 *>(s_rhs)[q] = reinterpret_cast<const d2 *>(A.rhs + base)[x];
      reinterpret_cast<d2 *>(s_tmp)[q] = reinterpret_cast<const d2 *>(A.tmp + base)[x];
    }
  }
  const double lambda2 = A.lambda2;
  // box position p of a level: its coordinate along d
  auto coord = [](int p, int lvl, int d) { return (p >> (d * (lvl - 1))) & ((1 << (lvl - 1)) - 1); };
  auto rhs_of = [&](int slot) {
    return TG::LOW && slot < TG::LOW ? s_rhs + slot * NCELL : A.rhs + (size_t)(s_id[slot] - 1) * NCELL;
  };
  auto tmp_of = [&](int slot) {
    return TG::LOW && slot < TG::LOW ? s_tmp + slot * NCELL : A.tmp + (size_t)(s_id[slot] - 1) * NCELL;
  };
  __syncthreads();

  // Edges (3D) and corners of a level's boxes, the faces being filled: the
  // diagonal neighbour's cell, or extrapolated from the face ghosts and the
  // box's own cells (as gc_box forms them).
  auto corners = [&](int o, int n_box) {
    for (int q = tid; q < n_box * NX; q += TAIL_NT) {
      const unsigned w = s_cr[o * NX + q];
      double *s = s_phi + (w & 0x3fff);
      if (w >> 31) {
        *s = s_phi[(w >> 14) & 0x3fff];
        continue;
      }
      // inwards along each axis
      const int ex = (w >> 14) & 3, ey = (w >> 16) & 3, ez = (w >> 18) & 3;
      const int di = ex == 0 ? 0 : ex == 1 ? 1 : -1, dj = (ey == 0 ? 0 : ey == 1 ? 1 : -1) * G::NG,
                dk = (ez == 0 ? 0 : ez == 1 ? 1 : -1) * G::NG * G::NG;
      if (D == 2) {
        *s = s[di] + s[dj] - s[di + dj];
      } else if (!ex || !ey || !ez) {
        // an edge along axis dim: the ghost moved inwards along axis
        // dim + 1, then the one along dim + 2
        const int g0 = !ex ? dj : !ey ? dk : di, g1 = !ex ? dk : !ey ? di : dj;
        *s = s[g0] + s[g1] - s[di + dj + dk];
      } else {
        *s = s[dj + dk] + s[di + dk] + s[di + dj] - 2 * s[di + dj + dk];
      }
    }
    __syncthreads();
  };
  // Face ghost w of a level: the neighbour's cell, or phys_ghost's sum.
  auto ghost_fill = [&](unsigned w, int lvl) {
    const int gd = w & 0x3fff, gs = (w >> 14) & 0x3fff;
    const double x1 = s_phi[gs];
    if (w >> 28 == TG_COPY) {
      s_phi[gd] = x1;
    } else {
      const double *bc = s_bc[lvl - 1][w >> 28];
      s_phi[gd] = bc[0] + bc[1] * x1 + 0.0 * s_phi[2 * gs - gd];
    }
  };
  // L phi at interior cell x (column col over all levels) of a box u
  auto apply = [&](const double *u, int x, const double *st, int col) {
    constexpr int sy = G::NG, sz = G::NG * G::NG;
    if (D == 2) {
      if (cyl) {
        const double *c = s_cyl[col];
        return c[0] * u[x] + c[1] * u[x - 1] + c[2] * u[x + 1] + st[3] * u[x - sy] + st[4] * u[x + sy];
      }
      return st[0] * u[x] + st[1] * u[x - 1] + st[2] * u[x + 1] + st[3] * u[x - sy] + st[4] * u[x + sy];
    }
    return st[0] * u[x] + st[1] * u[x - 1] + st[2] * u[x + 1] + st[3] * u[x - sy] + st[4] * u[x + sy] +
           st[5] * u[x - sz] + st[6] * u[x + sz];
  };

  for (int n_op = 0; n_op < A.n_ops; n_op++) {
    const TailOp op = A.ops[n_op];
    const int lvl = op.lvl, o = level_off(lvl), n_box = 1 << (D * (lvl - 1));
    const double *st = s_st[lvl - 1];
    // the first column of box p over all levels
    const int col0 = NC * ((1 << (lvl - 1)) - 1);
    auto col = [&](int p) { return col0 + NC * coord(p, lvl, 0); };
    switch (op.op) {
      case TL_SWEEP: {
        // What a thread's cells and ghosts need, once for all half-sweeps:
        // cell index, rhs and coefficients per colour, and the ghosts' words.
        double cs[7];
        for (int q = 0; q <= 2 * D; q++) cs[q] = st[q];
        const double inv_c0 = st[7];
        int cx[2][PER];
        unsigned gw[2][GPER];
        double rr[2][PER], k2[2][PER], k3[2][PER], ki[2][PER];
#pragma unroll
        for (int c = 0; c < 2; c++) {
#pragma unroll
          for (int t = 0; t < PER; t++) {
            const int q = tid + t * TAIL_NT;
            cx[c][t] = -1;
            rr[c][t] = k2[c][t] = k3[c][t] = ki[c][t] = 0;
            if (q < n_box * HALF) {
              const int p = q / HALF, r = q % HALF;
              const int j = (r / (NC / 2)) % NC + 1, k = (D == 3) ? r / ((NC / 2) * NC) + 1 : 0;
              const int i = 2 - ((c ^ (D == 3 ? k + j : j)) & 1) + 2 * (r % (NC / 2));
              cx[c][t] = (o + p) * NCELL + G::idx(i, j, k);
              rr[c][t] = rhs_of(o + p)[G::idx(i, j, k)];
              if (D == 2 && cyl) {
                const double *cc = s_cyl[col(p) + i - 1];
                k2[c][t] = cc[1];
                k3[c][t] = cc[2];
                ki[c][t] = cc[3];
              }
            }
          }
#pragma unroll
          for (int t = 0; t < GPER; t++) {
            const int q = tid + t * TAIL_NT, p = q / NGB;
            gw[c][t] = q < n_box * NGB ? s_gh[((o + p) * 2 + c) * NGB + q % NGB] : 0u;
          }
        }
        auto fill_ghosts = [&](auto C) {
          constexpr int c = decltype(C)::value;
#pragma unroll
          for (int t = 0; t < GPER; t++)
            if (tid + t * TAIL_NT < n_box * NGB) ghost_fill(gw[c][t], lvl);
        };
        auto half = [&](auto C, bool fill) {
          constexpr int c = decltype(C)::value;
          if (fill) {
            fill_ghosts(C);
            __syncthreads();
          }
#pragma unroll
          for (int t = 0; t < PER; t++) {
            if (cx[c][t] < 0) continue;
            constexpr int sy = G::NG, sz = G::NG * G::NG;
            double *s = s_phi + cx[c][t];
            const double rx = rr[c][t];
            if (D == 2) {
              if (cyl)
                s[0] = (rx - k2[c][t] * s[-1] - k3[c][t] * s[1] - cs[3] * s[-sy] - cs[4] * s[sy]) * ki[c][t];
              else
                s[0] = (rx - cs[1] * s[-1] - cs[2] * s[1] - cs[3] * s[-sy] - cs[4] * s[sy]) * inv_c0;
            } else {
              s[0] = (rx - cs[1] * s[-1] - cs[2] * s[1] - cs[3] * s[-sy] - cs[4] * s[sy] - cs[5] * s[-sz] -
                      cs[6] * s[sz]) *
                     inv_c0;
            }
          }
          __syncthreads();
        };
        for (int n = 1; n <= op.a; n += 2) {
          half(std::integral_constant<int, 1>(), !((op.b & TS_STORED) && n == 1));
          if (n < op.a) half(std::integral_constant<int, 0>(), true);
        }
        if (op.b & TS_GC) {
          fill_ghosts(std::integral_constant<int, 0>());
          fill_ghosts(std::integral_constant<int, 1>());
          __syncthreads();
        }
        if (op.b & TS_CORNERS) corners(o, n_box);
        break;
      }
      case TL_GC: {
        for (int q = tid; q < n_box * 2 * NGB; q += TAIL_NT) ghost_fill(s_gh[o * 2 * NGB + q], lvl);
        __syncthreads();
        if (op.a) corners(o, n_box);
        break;
      }
      case TL_RESTRICT:
        if constexpr (TG::LT > 1) {
          const int po = level_off(lvl - 1);
          for (int q = tid; q < n_box * NQ; q += TAIL_NT) {
            const int p = q / NQ, r = q % NQ;
            int pp = 0, off[3] = {0, 0, 0};
#pragma unroll
            for (int d = 0; d < D; d++) {
              const int c = coord(p, lvl, d);
              pp += (c >> 1) << (d * (lvl - 2));
              off[d] = (c & 1) * H;
            }
            const double *u = s_phi + (o + p) * NCELL, *rc = rhs_of(o + p);
            double *tc = tmp_of(o + p);
            const int i = r % H + 1, j = (r / H) % H + 1, k = (D == 3) ? r / (H * H) + 1 : 0;
            const int x0 = G::idx(2 * i - 1, 2 * j - 1, (D == 3) ? 2 * k - 1 : 0), c0 = col(p) + 2 * i - 2;
            // the children's residuals and values, in af_restrict_box's order
            double rs[4], sm = 0, sp = 0;
#pragma unroll
            for (int c = 0; c < NCH; c++) {
              const int x = x0 + (c & 1) + ((c >> 1) & 1) * G::NG + ((c >> 2) & 1) * G::NG * G::NG;
              const double rv = rc[x] - apply(u, x, st, c0 + (c & 1));
              if (op.a) tc[x] = rv;
              if (D == 2) rs[c & 3] = rv;
              sm = c ? sm + rv : rv;
              sp = c ? sp + u[x] : u[x];
            }
            const int ic = off[0] + i, y = G::idx(ic, off[1] + j, (D == 3) ? off[2] + k : 0);
            if (D == 2 && cyl) {
              // (the parent's column)
              const double tw = s_cyl[NC * ((1 << (lvl - 2)) - 1) + NC * coord(pp, lvl - 1, 0) + ic - 1][4];
              const double w1 = 1.0 - tw, w2 = 1.0 + tw;
              sm = w1 * (rs[0] + rs[2]) + w2 * (rs[1] + rs[3]);
            }
            tmp_of(po + pp)[y] = (1.0 / NCH) * sm;
            s_phi[(po + pp) * NCELL + y] = (1.0 / NCH) * sp;
          }
          __syncthreads();
        }
        break;
      case TL_RHS: {
        for (int q = tid; q < n_box * NCELL; q += TAIL_NT) {
          const int p = q / NCELL, x = q % NCELL;
          if (!s_par[o + p]) continue;
          const double *u = s_phi + (o + p) * NCELL;
          double *r = rhs_of(o + p) + x, *t = tmp_of(o + p) + x;
          const int i = x % G::NG, j = (x / G::NG) % G::NG, k = (D == 3) ? x / (G::NG * G::NG) : 0;
          const bool inner = i >= 1 && i <= NC && j >= 1 && j <= NC && (D == 2 || (k >= 1 && k <= NC));
          const double rv = inner ? apply(u, x, st, col(p) + i - 1) : *r;
          *r = rv + *t;
          if (op.a) *t = u[x];
        }
        __syncthreads();
        break;
      }
      case TL_SOLVE: {
        Sten<D, double> sten;
        for (int q = 0; q <= 2 * D; q++) sten.c[q] = st[q];
        const DBox &b1 = A.boxes[__builtin_amdgcn_readfirstlane(s_id[0]) - 1];
        const double *r = rhs_of(0);
        for (int q = tid; q < G::NINT; q += TAIL_NT) {
          int i, j, k;
          interior_ijk<D, NC>(q, i, j, k);
          s_buf[q] = coarse_rhs_value<D, NC>(b1, A.m, sten, cyl, r[G::idx(i, j, k)], i, j, k);
        }
        __syncthreads();
        coarse_transforms<D, NC, TAIL_NT>(s_buf, s_mat, s_mat + NMAT, lambda2);
        for (int q = tid; q < G::NINT; q += TAIL_NT) {
          int i, j, k;
          interior_ijk<D, NC>(q, i, j, k);
          s_phi[G::idx(i, j, k)] = s_buf[q];
        }
        __syncthreads();
        break;
      }
      case TL_COPY:
      case TL_SUB: {
        for (int q = tid; q < n_box * NCELL; q += TAIL_NT) {
          const int p = q / NCELL, x = q % NCELL;
          double *t = tmp_of(o + p) + x;
          const double v = s_phi[(o + p) * NCELL + x];
          if (op.op == TL_COPY)
            *t = v;
          else if (s_par[o + p])
            *t = v - *t;
        }
        __syncthreads();
        break;
      }
      case TL_PROLONG:
        if constexpr (TG::LT > 1) {
          const int po = level_off(lvl - 1);
          for (int q = tid; q < n_box * G::NINT; q += TAIL_NT) {
            const int p = q / G::NINT;
            int i, j, k;
            interior_ijk<D, NC>(q % G::NINT, i, j, k);
            int pp = 0, off[3] = {0, 0, 0};
#pragma unroll
            for (int d = 0; d < D; d++) {
              const int c = coord(p, lvl, d);
              pp += (c >> 1) << (d * (lvl - 2));
              off[d] = (c & 1) * H;
            }
            double &u = s_phi[(o + p) * NCELL + G::idx(i, j, k)];
            // (level - 1 is below the finest held: its tmp is in LDS)
            u = prolong_value<D, NC, double>(u, s_tmp + (po + pp) * NCELL, off, i, j, k);
          }
          __syncthreads();
        }
        break;
      case TL_RESID: {
        double mx = 0;
        for (int q = tid; q < n_box * G::NINT; q += TAIL_NT) {
          const int p = q / G::NINT;
          int i, j, k;
          interior_ijk<D, NC>(q % G::NINT, i, j, k);
          const int x = G::idx(i, j, k);
          const double lp = apply(s_phi + (o + p) * NCELL, x, st, col(p) + i - 1);
          const double rv = rhs_of(o + p)[x] - lp;
          tmp_of(o + p)[x] = rv;
          if (!s_par[o + p]) mx = fmax(mx, fabs(rv));
        }
        for (int f = 32; f > 0; f >>= 1) mx = fmax(mx, __shfl_xor(mx, f));
        if ((tid & 63) == 0 && mx > 0) atomic_max_nonneg(A.red + (size_t)run * RED_STRIPES * RED_STRIDE, mx);
        __syncthreads();
        break;
      }
      case TL_RESET: {
        if (tid < RED_STRIPES) A.red[((size_t)run * RED_STRIPES + tid) * RED_STRIDE] = 0ull;
        __syncthreads();
        break;
      }
    }
  }
  for (int q = tid; q < n_slots * NV; q += TAIL_NT) {
    const int s = q / NV, x = q - s * NV;
    const size_t base = (size_t)(s_id[s] - 1) * NCELL;
    reinterpret_cast<d2 *>(A.phi + base)[x] = reinterpret_cast<const d2 *>(s_phi)[q];
    if (TG::LOW && s < n_low) {
      reinterpret_cast<d2 *>(A.rhs + base)[x] = reinterpret_cast<const d2 *>(s_rhs)[q];
      reinterpret_cast<d2 *>(A.tmp + base)[x] = reinterpret_cast<const d2 *>(s_tmp)[q];
    }
  }
}

}  // namespace afg
