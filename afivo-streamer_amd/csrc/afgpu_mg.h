// Multigrid and ghost-cell kernels (afivo/src/m_af_multigrid.f90,
// m_af_stencil.f90, m_af_ghostcell.f90, m_af_restrict.f90).
//
// Work decomposition: a launch covers a box list; each box is handled by
// `bpb` workgroups ("blocks per box", > 1 on the coarse levels that have few
// boxes, so that those launches still spread over the CUs).  Every cell
// value is computed with the reference's operation order, so the FP64
// instantiation reproduces the CPU path bit for bit (hipcc is run with
// -ffp-contract=off).  The same templates instantiated with T = float form
// the inner cycle of the mixed-precision solver.
#pragma once

#include "afgpu_common.h"

namespace afg {

// Box of work item w (box w / bpb, part w % bpb) and the first cell index /
// stride of this thread.
struct Part {
  int id;
  int q0;
  int stride;
};
template <int BS>
__device__ inline Part part_of(const int *__restrict__ ids, int bpb, int w) {
  Part p;
  const int slot = w / bpb;
  p.id = ids[slot];
  p.q0 = (w - slot * bpb) * BS + ltid<BS>();
  p.stride = bpb * BS;
  return p;
}

// Constant 3/5/7-point stencil of a box (mg_box_lpl_stencil,
// afivo/src/m_af_multigrid.f90:1246-1264).
template <int D, typename T>
struct Sten {
  T c[7];
};
template <int D, typename T>
__device__ inline Sten<D, T> lpl_stencil(const DBox &bx, T lambda2) {
  Sten<D, T> s;
  for (int d = 0; d < D; d++) {
    T dr = (T)bx.dr[d];
    T inv_dr2 = T(1) / (dr * dr);
    s.c[1 + 2 * d] = inv_dr2;
    s.c[2 + 2 * d] = inv_dr2;
  }
  T sum = T(0);
  for (int q = 1; q <= 2 * D; q++) sum = sum + s.c[q];
  s.c[0] = -sum - lambda2;
  return s;
}

// Per-i cylindrical coefficients (af_cyl_flux_factors m_af_types.f90:1199
// and the cc_cyl construction of m_af_stencil.f90:388-394, 871-877).
template <typename T>
__device__ inline void cyl_coeffs(const DBox &bx, int i, const T *c, T &c1, T &c2, T &c3) {
  T dr = (T)bx.dr[0];
  T r = (T)bx.r_min[0] + (T(i) - T(0.5)) * dr;
  T inv_r = T(1) / r;
  T rf1 = (r - T(0.5) * dr) * inv_r;
  T rf2 = (r + T(0.5) * dr) * inv_r;
  c2 = rf1 * c[1];
  c3 = rf2 * c[2];
  c1 = c[0] - (c2 - c[1]) - (c3 - c[2]);
}

// L phi at interior cell (i,j,k) (stencil_apply_357, m_af_stencil.f90:367-496)
// of a box stored with layout L (afivo's by default: LDS copies, FP64 pools).
template <int D, int NC, typename T, typename L = LayStd<D, NC>>
__device__ inline T apply_cell(const T *u, const Sten<D, T> &s, bool cyl, const DBox &bx, int i, int j, int k) {
  using G = Geo<D, NC>;
  if constexpr (L::SPLIT) {
    const T uc = u[L::in_at(i, j, k)], xm = u[L::nb_at(i, j, k, 0, -1)], xp = u[L::nb_at(i, j, k, 0, 1)];
    const T ym = u[L::nb_at(i, j, k, 1, -1)], yp = u[L::nb_at(i, j, k, 1, 1)];
    if (D == 2) {
      if (cyl) {
        T c1, c2, c3;
        cyl_coeffs<T>(bx, i, s.c, c1, c2, c3);
        return c1 * uc + c2 * xm + c3 * xp + s.c[3] * ym + s.c[4] * yp;
      }
      return s.c[0] * uc + s.c[1] * xm + s.c[2] * xp + s.c[3] * ym + s.c[4] * yp;
    }
    return s.c[0] * uc + s.c[1] * xm + s.c[2] * xp + s.c[3] * ym + s.c[4] * yp + s.c[5] * u[L::nb_at(i, j, k, 2, -1)] +
           s.c[6] * u[L::nb_at(i, j, k, 2, 1)];
  }
  const int x = G::idx(i, j, k);
  if (D == 2) {
    if (cyl) {
      T c1, c2, c3;
      cyl_coeffs<T>(bx, i, s.c, c1, c2, c3);
      return c1 * u[x] + c2 * u[x - 1] + c3 * u[x + 1] + s.c[3] * u[x - G::NG] + s.c[4] * u[x + G::NG];
    }
    return s.c[0] * u[x] + s.c[1] * u[x - 1] + s.c[2] * u[x + 1] + s.c[3] * u[x - G::NG] +
           s.c[4] * u[x + G::NG];
  } else {
    constexpr int NG2 = G::NG * G::NG;
    return s.c[0] * u[x] + s.c[1] * u[x - 1] + s.c[2] * u[x + 1] + s.c[3] * u[x - G::NG] +
           s.c[4] * u[x + G::NG] + s.c[5] * u[x - NG2] + s.c[6] * u[x + NG2];
  }
}

template <int D, int NC>
__device__ inline void interior_ijk(int q, int &i, int &j, int &k) {
  i = q % NC + 1;
  j = (q / NC) % NC + 1;
  k = (D == 3) ? q / (NC * NC) + 1 : 0;
}

// ---- ghost cells --------------------------------------------------------------
// Value of the ghost cell of face nb at tangential position (a, b) of box
// `id`, as af_gc_box (afivo/src/m_af_ghostcell.f90:64-120) sets it: copy of
// the same-level neighbour (copy_from_nb :654), physical boundary (bc_to_gc
// :173-279), or refinement boundary (mg_sides_rb, m_af_multigrid.f90:294-461,
// or af_gc_interp / af_gc_interp_lim, m_af_ghostcell.f90:394-605).  x1 and x2
// are the box's first and second interior cells along the face normal.
// `coarse` (default: var) holds the coarser level's values when the box's
// own level is kept in a different buffer.
// The part of a ghost value of a face without a same-level neighbour
// (nb_id <= 0) that does not depend on the box's own cells: the boundary
// value's term, or the coarse interpolation at a refinement boundary (and
// the coarse cell the limiter compares with).  ghost_finish() adds the
// terms of the box's cells x1, x2 in the order ghost_value() always used.
template <typename T>
struct GhostPart {
  T p, c1;
};
// ghost_coarse in two phases: the coarse values it reads (none on a
// physical boundary), then the part formed from them, so that a kernel can
// have the loads of several ghosts in flight before it forms any.
template <typename T>
struct CoarseVals {
  T v[5];
};
template <int D, int NC, typename T>
__device__ inline CoarseVals<T> ghost_coarse_load(const DBox &bx, const T *var, const VarBc &m, int nb, int a, int b,
                                                  const T *coarse = nullptr) {
  using L = Lay<D, NC, T>;
  constexpr int H = NC / 2;
  const int d = nb / 2;
  const bool low = (nb % 2) == 0;
  int t0, t1;
  tangential(D, d, t0, t1);
  CoarseVals<T> cv = {{T(0), T(0), T(0), T(0), T(0)}};
  if (bx.nb[nb] < 0) return cv;
  const T *P = (coarse ? coarse : var) + (size_t)(bx.pnb[nb] - 1) * L::STRIDE;
  int co[3] = {0, 0, 0};
  for (int dd = 0; dd < D; dd++) co[dd] = ((bx.ix[dd] - 1) & 1) * H;
  // coarse cell at tangential (qa, qb) on the coarse neighbour's face cn
  auto at = [&](int cn, int qa, int qb) {
    int q[3] = {0, 0, 0};
    q[d] = cn;
    q[t0] = qa;
    if (D == 3) q[t1] = qb;
    return P[L::at(q[0], q[1], q[2])];
  };
  const int cn = low ? NC : 1;
  if (m.rb == RB_MG) {
    const int i = (a + 1) >> 1, j = (b + 1) >> 1;
    if (D == 2) {
      cv.v[0] = at(cn, co[t0] + i + 1, 0);
      cv.v[1] = at(cn, co[t0] + i - 1, 0);
      cv.v[2] = at(cn, co[t0] + i, 0);
    } else {
      cv.v[0] = at(cn, co[t0] + i + 1, co[t1] + j);
      cv.v[1] = at(cn, co[t0] + i - 1, co[t1] + j);
      cv.v[2] = at(cn, co[t0] + i, co[t1] + j + 1);
      cv.v[3] = at(cn, co[t0] + i, co[t1] + j - 1);
      cv.v[4] = at(cn, co[t0] + i, co[t1] + j);
    }
    return cv;
  }
  const int a1 = co[t0] + ((a + 1) >> 1), a2 = a1 + 1 - 2 * (a & 1);
  if (D == 2) {
    cv.v[0] = at(cn, a1, 0);
    cv.v[1] = at(cn, a2, 0);
  } else {
    const int b1 = co[t1] + ((b + 1) >> 1), b2 = b1 + 1 - 2 * (b & 1);
    cv.v[0] = at(cn, a1, b1);
    cv.v[1] = at(cn, a2, b1);
    cv.v[2] = at(cn, a1, b2);
  }
  return cv;
}
// The part of a refinement-boundary ghost formed from the coarse values.
template <int D, typename T>
__device__ inline GhostPart<T> coarse_part(const VarBc &m, int d, int a, int b, const CoarseVals<T> &cv) {
  GhostPart<T> g;
  g.c1 = T(0);
  if (m.rb == RB_MG) {
    if (D == 2) {
      const T grad = T(0.125) * (cv.v[0] - cv.v[1]);
      g.p = (a & 1) ? cv.v[2] - grad : cv.v[2] + grad;
    } else {
      const T g1 = T(0.125) * (cv.v[0] - cv.v[1]);
      const T g2 = T(0.125) * (cv.v[2] - cv.v[3]);
      const T tc = cv.v[4];
      const T h = (a & 1) ? tc - g1 : tc + g1;
      g.p = (b & 1) ? h - g2 : h + g2;
    }
    return g;
  }
  const T third = T(1 / 3.0), sixth = T(1 / 6.0);
  if (D == 2) {
    g.p = T(0.5) * cv.v[0] + sixth * cv.v[1];
  } else {
    // the z-face case sums the off-diagonal coarse values in the other order
    const T c2 = (d == 2) ? cv.v[2] : cv.v[1], c3 = (d == 2) ? cv.v[1] : cv.v[2];
    g.p = third * cv.v[0] + sixth * c2 + sixth * c3;
  }
  g.c1 = cv.v[0];
  return g;
}
// ... and the terms of the box's cells x1, x2.
template <typename T>
__device__ inline T rb_finish(const VarBc &m, const GhostPart<T> &g, T x1, T x2) {
  if (m.rb == RB_MG) return T(0.5) * g.p + T(0.75) * x1 - T(0.25) * x2;
  T v = g.p + T(1 / 3.0) * x1;
  if (m.rb == RB_INTERP_LIM && v > 2 * g.c1) v = 2 * g.c1;
  return v;
}
template <int D, int NC, typename T>
__device__ inline GhostPart<T> ghost_coarse_form(const DBox &bx, const VarBc &m, int nb, int a, int b,
                                                 const CoarseVals<T> &cv) {
  const int d = nb / 2;
  const bool low = (nb % 2) == 0;
  GhostPart<T> g;
  g.c1 = T(0);
  if (bx.nb[nb] < 0) {
    T c0;
    if (m.type[nb] == BC_DIRICHLET)
      c0 = 2;
    else if (m.type[nb] == BC_NEUMANN)
      c0 = (T)bx.dr[d] * T(low ? -1 : 1);
    else
      c0 = 1;
    g.p = c0 * (T)bc_value(m, nb, bx.run);
    return g;
  }
  return coarse_part<D, T>(m, d, a, b, cv);
}
template <int D, int NC, typename T>
__device__ inline GhostPart<T> ghost_coarse(const DBox &bx, const T *var, const VarBc &m, int nb, int a, int b,
                                            const T *coarse = nullptr) {
  return ghost_coarse_form<D, NC, T>(bx, m, nb, a, b, ghost_coarse_load<D, NC, T>(bx, var, m, nb, a, b, coarse));
}

template <int D, int NC, typename T>
__device__ inline T ghost_finish(const DBox &bx, const VarBc &m, int nb, const GhostPart<T> &g, T x1, T x2) {
  if (bx.nb[nb] < 0) {
    T c1, c2;
    if (m.type[nb] == BC_DIRICHLET) {
      c1 = -1; c2 = 0;
    } else if (m.type[nb] == BC_NEUMANN) {
      c1 = 1; c2 = 0;
    } else {
      c1 = 0; c2 = 0;
    }
    return g.p + c1 * x1 + c2 * x2;
  }
  return rb_finish<T>(m, g, x1, x2);
}

template <int D, int NC, typename T>
__device__ inline T ghost_value(const DBox *__restrict__ boxes, const DBox &bx, const T *var, const VarBc &m, int nb,
                                int a, int b, T x1, T x2, const T *coarse = nullptr) {
  using L = Lay<D, NC, T>;
  const int d = nb / 2;
  const bool low = (nb % 2) == 0;
  int t0, t1;
  tangential(D, d, t0, t1);
  const int nb_id = bx.nb[nb];
  if (nb_id > 0) {
    const T *w = var + (size_t)(nb_id - 1) * L::STRIDE;
    int q[3] = {0, 0, 0};
    q[t0] = a;
    if (D == 3) q[t1] = b;
    q[d] = low ? NC : 1;
    return w[L::at(q[0], q[1], q[2])];
  }
  return ghost_finish<D, NC, T>(bx, m, nb, ghost_coarse<D, NC, T>(bx, var, m, nb, a, b, coarse), x1, x2);
}

// Position of face cell (nb, a, b) at normal index p.
template <int D>
__device__ inline void face_pos(int nb, int a, int b, int pn, int *p) {
  const int d = nb / 2;
  int t0, t1;
  tangential(D, d, t0, t1);
  p[0] = p[1] = p[2] = 0;
  p[t0] = a;
  if (D == 3) p[t1] = b;
  p[d] = pn;
}

// tmp = rhs - L phi on interior cells (residual_box, m_af_multigrid.f90:801-810);
// for leaf boxes the max |tmp| is also reduced into *leafmax
// (af_tree_maxabs_cc, afivo/src/m_af_utils.f90:773).
template <int D, int NC, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_residual(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                      const T *__restrict__ phi, const T *__restrict__ rhs, T *tmp,
                                                      T lambda2, int cyl, unsigned long long *leafmax, int bpb,
                                                      int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  __shared__ double sh[BS / 64];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const int id = pt.id;
    const DBox &bx = boxes[id - 1];
    const Sten<D, T> s = lpl_stencil<D, T>(bx, lambda2);
    const size_t base = (size_t)(id - 1) * L::STRIDE;
    double mx = 0;
    for (int q = pt.q0; q < G::NINT; q += pt.stride) {
      int i, j, k;
      interior_ijk<D, NC>(q, i, j, k);
      const int x = L::in_at(i, j, k);
      T lp = apply_cell<D, NC, T, L>(phi + base, s, cyl != 0, bx, i, j, k);
      const T rv = rhs[base + x] - lp;
      tmp[base + x] = rv;
      mx = fmax(mx, (double)fabs(rv));
    }
    if (leafmax && bx.children[0] == 0) {
      mx = group_max<BS, BB>(mx, sh);
      if (ltid<BS>() == 0) atomic_max_nonneg(run_slot(leafmax, bx), mx);
    }
  }
}

// Positions in layout L of the 2^D children cells of a parent cell:
// child c is (i_f + (c & 1), jf + ((c >> 1) & 1), kf + ((c >> 2) & 1)),
// with i_f, jf (and kf) odd.  (In the colour-split layout the first cell
// of each pair of the x direction is at an even lexicographic index, so both
// share one position within their colour blocks.)
template <int D, int NC, typename L>
__host__ __device__ inline void child_pos(int i_f, int jf, int kf, int *pos) {
  constexpr int nch = (D == 3) ? 8 : 4;
  if constexpr (L::SPLIT) {
    const int h0 = ((i_f - 1) + NC * ((jf - 1) + NC * (D == 3 ? kf - 1 : 0))) >> 1;
    const int col0 = (i_f + jf + kf) & 1;
    for (int c = 0; c < nch; c++) {
      const int di = c & 1, dj = (c >> 1) & 1, dk = (c >> 2) & 1;
      pos[c] = ((col0 + di + dj + dk) & 1) * L::HALF + h0 + dj * (NC / 2) + dk * (NC * NC / 2);
    }
  } else {
    for (int c = 0; c < nch; c++) pos[c] = L::in_at(i_f + (c & 1), jf + ((c >> 1) & 1), kf + ((c >> 2) & 1));
  }
}

// Cylindrical weight of a parent cell's restriction.
template <typename T>
__device__ inline T restrict_weight(const DBox &bp, int ic) {
  const T r = (T)bp.r_min[0] + (T(ic) - T(0.5)) * (T)bp.dr[0];
  return T(0.25) * (T)bp.dr[0] / r;
}

// Restriction of one parent cell from its 2^D children values
// (af_restrict_box, afivo/src/m_af_restrict.f90:62-136).
template <int D, int NC, typename T, typename L = LayStd<D, NC>>
__device__ inline T restrict_cell(const T *f, int i_f, int jf, int kf, bool cyl_geom, const DBox &bp, int ic) {
  int p[8];
  child_pos<D, NC, L>(i_f, jf, kf, p);
  if (D == 2) {
    if (cyl_geom) {
      const T t = restrict_weight<T>(bp, ic);
      T w1 = T(1) - t, w2 = T(1) + t;
      return T(0.25) * (w1 * (f[p[0]] + f[p[2]]) + w2 * (f[p[1]] + f[p[3]]));
    }
    T s = f[p[0]];
    s = s + f[p[1]];
    s = s + f[p[2]];
    s = s + f[p[3]];
    return T(0.25) * s;
  } else {
    T s = f[p[0]];
    for (int c = 1; c < 8; c++) s = s + f[p[c]];
    return T(0.125) * s;
  }
}

// Restrict variable `src` of child boxes into `dst` of their parents.
template <int D, int NC, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_restrict(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                      const T *src, T *dst, int use_geom, int cyl, int bpb, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  constexpr int H = NC / 2;
  constexpr int NQ = (D == 3) ? H * H * H : H * H;
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const int id = pt.id;
    const DBox &bc = boxes[id - 1];
    const DBox &bp = boxes[bc.parent - 1];
    int off[3] = {0, 0, 0};
    for (int d = 0; d < D; d++) off[d] = ((bc.ix[d] - 1) & 1) * H;
    const T *f = src + (size_t)(id - 1) * L::STRIDE;
    T *u = dst + (size_t)(bc.parent - 1) * L::STRIDE;
    for (int q = pt.q0; q < NQ; q += pt.stride) {
      const int i = q % H + 1, j = (q / H) % H + 1, k = (D == 3) ? q / (H * H) + 1 : 0;
      const int ic = off[0] + i, jc = off[1] + j, kc = (D == 3) ? off[2] + k : 0;
      u[L::at(ic, jc, kc)] =
          restrict_cell<D, NC, T, L>(f, 2 * i - 1, 2 * j - 1, (D == 3) ? 2 * k - 1 : 0, cyl && use_geom, bp, ic);
    }
  }
}

// update_coarse / set_coarse_phi_rhs, second half (m_af_multigrid.f90:726-736):
// on parents, rhs = L phi (interior) + tmp (all cells); optionally tmp = phi.
template <int D, int NC, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_coarse_rhs(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                        const T *__restrict__ phi, T *rhs, T *tmp, T lambda2, int cyl,
                                                        int copy_phi, int bpb, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const int id = pt.id;
    const DBox &bx = boxes[id - 1];
    const Sten<D, T> s = lpl_stencil<D, T>(bx, lambda2);
    const size_t base = (size_t)(id - 1) * L::STRIDE;
    for (int x = pt.q0; x < G::NCELL; x += pt.stride) {
      int i, j, k;
      bool inner;
      if constexpr (L::SPLIT) {
        inner = x < G::NINT;
        if (inner) colour_cell<D, NC>(x >= L::HALF, x >= L::HALF ? x - L::HALF : x, i, j, k);
      } else {
        i = x % G::NG, j = (x / G::NG) % G::NG, k = (D == 3) ? x / (G::NG * G::NG) : 0;
        inner = i >= 1 && i <= NC && j >= 1 && j <= NC && (D == 2 || (k >= 1 && k <= NC));
      }
      // (nothing reads the ghost part of a split pool's rhs)
      if (inner || !L::SPLIT) {
        const T rv = inner ? apply_cell<D, NC, T, L>(phi + base, s, cyl != 0, bx, i, j, k) : rhs[base + x];
        rhs[base + x] = rv + tmp[base + x];
      }
      if (copy_phi) tmp[base + x] = phi[base + x];
    }
  }
}

// Whole-box elementwise operations (afivo/src/m_af_utils.f90:385-576).
enum BoxOp { OP_COPY = 0, OP_CLEAR = 1, OP_SUB_FROM = 2, OP_AXPY_NEG = 3 };
// OP_COPY: b = a; OP_CLEAR: b = 0; OP_SUB_FROM: b = a - b; OP_AXPY_NEG: b = b - s*a
// A box's NCELL words are a whole number of 16-byte words (every box size
// here), so the operations run on 16-byte words: each lane moves 16 bytes
// per access.
template <typename T>
struct alignas(16) Word16 {
  T v[16 / sizeof(T)];
};
template <int NCELL, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_boxop(const int *__restrict__ ids, const T *a, T *b, int op, T s, int bpb,
                                                   int nw) {
  using V = Word16<T>;
  constexpr int NL = 16 / sizeof(T);
  static_assert((NCELL * sizeof(T)) % 16 == 0, "boxes of whole 16-byte words");
  constexpr int NV = NCELL / NL;
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const V *av = reinterpret_cast<const V *>(a + (size_t)(pt.id - 1) * NCELL);
    V *bv = reinterpret_cast<V *>(b + (size_t)(pt.id - 1) * NCELL);
    for (int x = pt.q0; x < NV; x += pt.stride) {
      V r;
      switch (op) {
        case OP_COPY: r = av[x]; break;
        case OP_CLEAR:
          for (int l = 0; l < NL; l++) r.v[l] = T(0);
          break;
        case OP_SUB_FROM: {
          const V p = av[x], q = bv[x];
          for (int l = 0; l < NL; l++) r.v[l] = p.v[l] - q.v[l];
          break;
        }
        default: {
          const V p = av[x], q = bv[x];
          for (int l = 0; l < NL; l++) r.v[l] = q.v[l] - s * p.v[l];
          break;
        }
      }
      bv[x] = r;
    }
  }
}

// v + P(tmp) at cell (i, j, k) of a child box at offset off within its
// parent, whose values P are: stencil_prolong_248
// (afivo/src/m_af_stencil.f90:695-815) with the weights of
// mg_box_prolong_linear_stencil (m_af_multigrid.f90:1267-1284).
template <int D, int NC, typename T>
__device__ inline T prolong_value(T v, const T *P, const int *off, int i, int j, int k) {
  using L = Lay<D, NC, T>;
  const int i1 = off[0] + ((i + 1) >> 1), i2 = i1 + 1 - 2 * (i & 1);
  const int j1 = off[1] + ((j + 1) >> 1), j2 = j1 + 1 - 2 * (j & 1);
  if (D == 2) {
    const T w0 = T(9 / 16.0), w1 = T(3 / 16.0), w2 = T(3 / 16.0), w3 = T(1 / 16.0);
    return v + w0 * P[L::at(i1, j1, 0)] + w1 * P[L::at(i2, j1, 0)] + w2 * P[L::at(i1, j2, 0)] +
           w3 * P[L::at(i2, j2, 0)];
  }
  const int k1 = off[2] + ((k + 1) >> 1), k2 = k1 + 1 - 2 * (k & 1);
  const T w0 = T(27 / 64.0), w1 = T(9 / 64.0), w3 = T(3 / 64.0), w7 = T(1 / 64.0);
  return v + w0 * P[L::at(i1, j1, k1)] + w1 * P[L::at(i2, j1, k1)] + w1 * P[L::at(i1, j2, k1)] +
         w3 * P[L::at(i2, j2, k1)] + w1 * P[L::at(i1, j1, k2)] + w3 * P[L::at(i2, j1, k2)] +
         w3 * P[L::at(i1, j2, k2)] + w7 * P[L::at(i2, j2, k2)];
}

// phi(child) += P(tmp(parent)), with add.
template <int D, int NC, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_prolong_add(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                         const T *__restrict__ src, T *dst, int bpb, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  constexpr int H = NC / 2;
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const int id = pt.id;
    const DBox &bc = boxes[id - 1];
    const T *P = src + (size_t)(bc.parent - 1) * L::STRIDE;
    T *u = dst + (size_t)(id - 1) * L::STRIDE;
    int off[3] = {0, 0, 0};
    for (int d = 0; d < D; d++) off[d] = ((bc.ix[d] - 1) & 1) * H;
    for (int q = pt.q0; q < G::NINT; q += pt.stride) {
      int i, j, k;
      interior_ijk<D, NC>(q, i, j, k);
      T &v = u[L::at(i, j, k)];
      v = prolong_value<D, NC, T>(v, P, off, i, j, k);
    }
  }
}

// k_prolong_add for pools in the colour-split layout: the parent cells the
// box's cells interpolate from (its octant and one cell around it) are
// staged in LDS once, then every cell is formed from LDS, colour block by
// colour block (same weights and order as k_prolong_add).  What is
// interpolated is the parent's change since the descent, phi - tmp, formed
// while it is staged: a pass of its own over the parents (which the FP64
// form keeps, its tmp being part of the state compared with the oracle) is
// a launch more in every level's visit.  A step of a 3D channel of 8^3
// boxes takes 13.4 ms instead of 13.7, of 16^3 boxes 22.8 instead of 23.1.
template <int D, int NC, int BS, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_prolong_add_split(const int *__restrict__ ids,
                                                               const DBox *__restrict__ boxes,
                                                               const float *phi, const float *__restrict__ tmp,
                                                               float *dst, int bpb, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, float>;
  constexpr int H = NC / 2, P = H + 2;
  constexpr int NP = (D == 3) ? P * P * P : P * P;
  __shared__ float s_all[BB][NP];
  float *sp = s_all[lgrp<BS, BB>()];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const DBox &bc = boxes[pt.id - 1];
    const size_t pb = (size_t)(bc.parent - 1) * L::STRIDE;
    float *u = dst + (size_t)(pt.id - 1) * L::STRIDE;
    int off[3] = {0, 0, 0};
    for (int d = 0; d < D; d++) off[d] = ((bc.ix[d] - 1) & 1) * H;
    // parent cells off[d] .. off[d] + H + 1 along each axis
    for (int q = ltid<BS>(); q < NP; q += BS) {
      const int a = q % P, b = (q / P) % P, c = (D == 3) ? q / (P * P) : 0;
      const int x = L::at(off[0] + a, off[1] + b, (D == 3) ? off[2] + c : 0);
      sp[q] = phi[pb + x] - tmp[pb + x];
    }
    gsync<BS, BB>();
    auto S = [&](int a, int b, int c) { return sp[a + P * (b + P * c)]; };
    for (int x = pt.q0; x < G::NINT; x += pt.stride) {
      int i, j, k;
      colour_cell<D, NC>(x >= L::HALF, x >= L::HALF ? x - L::HALF : x, i, j, k);
      const int i1 = (i + 1) >> 1, i2 = i1 + 1 - 2 * (i & 1);
      const int j1 = (j + 1) >> 1, j2 = j1 + 1 - 2 * (j & 1);
      if (D == 2) {
        const float w0 = 9 / 16.0f, w1 = 3 / 16.0f, w2 = 3 / 16.0f, w3 = 1 / 16.0f;
        u[x] = u[x] + w0 * S(i1, j1, 0) + w1 * S(i2, j1, 0) + w2 * S(i1, j2, 0) + w3 * S(i2, j2, 0);
      } else {
        const int k1 = (k + 1) >> 1, k2 = k1 + 1 - 2 * (k & 1);
        const float w0 = 27 / 64.0f, w1 = 9 / 64.0f, w3 = 3 / 64.0f, w7 = 1 / 64.0f;
        u[x] = u[x] + w0 * S(i1, j1, k1) + w1 * S(i2, j1, k1) + w1 * S(i1, j2, k1) + w3 * S(i2, j2, k1) +
               w1 * S(i1, j1, k2) + w3 * S(i2, j1, k2) + w3 * S(i1, j2, k2) + w7 * S(i2, j2, k2);
      }
    }
    gsync<BS, BB>();  // (the group's LDS is reused by its next item)
  }
}

// max |u| over interior cells of a box list (af_tree_maxabs_cc,
// afivo/src/m_af_utils.f90:773).
template <int D, int NC, int BS, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_maxabs(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                    const double *__restrict__ u, unsigned long long *out, int bpb,
                                                    int nw) {
  using G = Geo<D, NC>;
  __shared__ double sh[BS / 64];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const size_t base = (size_t)(pt.id - 1) * G::NCELL;
    double m = 0;
    for (int q = pt.q0; q < G::NINT; q += pt.stride) {
      int i, j, k;
      interior_ijk<D, NC>(q, i, j, k);
      m = fmax(m, fabs(u[base + G::idx(i, j, k)]));
    }
    m = group_max<BS, BB>(m, sh);
    if (ltid<BS>() == 0) atomic_max_nonneg(run_slot(out, boxes[pt.id - 1]), m);
  }
}

// Level-1 rhs b at cell (i, j, k) with the boundary values folded in, as
// coarse_solver_set_rhs_phi does (afivo/src/m_coarse_solver.f90:286-338).
template <int D, int NC>
__device__ inline double coarse_rhs_value(const DBox &bx, const VarBc &m, const Sten<D, double> &s, bool cyl, double b,
                                          int i, int j, int k) {
  const int p[3] = {i, j, (D == 3) ? k : 1};
#pragma unroll
  for (int nb = 0; nb < 2 * D; nb++) {
    if (bx.nb[nb] >= 0) continue;
    const int d = nb / 2;
    const bool low = (nb % 2) == 0;
    if (p[d] != (low ? 1 : NC)) continue;
    double cnb = s.c[1 + nb];
    if (cyl && d == 0) {
      double dr = bx.dr[0];
      double rr = bx.r_min[0] + (i - 0.5) * dr;
      double inv_r = 1 / rr;
      double rf = low ? (rr - 0.5 * dr) * inv_r : (rr + 0.5 * dr) * inv_r;
      cnb = rf * s.c[1 + nb];
    }
    double f;
    if (m.type[nb] == BC_DIRICHLET)
      f = -2 * cnb;
    else
      f = -(cnb * bx.dr[d]) * (double)(low ? -1 : 1);
    b = b + f * bc_value(m, nb, bx.run);
  }
  return b;
}
// One axis of the level-1 transforms: out = M buf along axis AX, with M's
// rows padded to NC + 1 (rows of different lanes then lie in different LDS
// banks).  A thread's cells differ along the last axis, so along the other
// axes they share the matrix row and along the last axis the line.
template <int D, int NC, int NT, int AX>
__device__ inline void coarse_axis(double *buf, const double *M) {
  constexpr int N = Geo<D, NC>::NINT, PER = (N + NT - 1) / NT;
  constexpr int st = (AX == 0) ? 1 : (AX == 1) ? NC : NC * NC;
  static_assert(N % NT == 0 || N < NT, "whole strides of cells");
  const int tid = threadIdx.x;
  double out[PER];
  if (tid < N) {
    int row[PER], line[PER];
#pragma unroll
    for (int t = 0; t < PER; t++) {
      const int q = tid + t * NT;
      row[t] = (q / st) % NC;
      line[t] = q - row[t] * st;
      out[t] = 0.0;
    }
    if constexpr (AX < D - 1 && N > NT) row[PER - 1] = row[0];  // (equal; so the compiler reads the row once)
#pragma unroll 4
    for (int mm = 0; mm < NC; mm++) {
      const double m0 = M[row[0] * (NC + 1) + mm], b0 = buf[line[0] + mm * st];
#pragma unroll
      for (int t = 0; t < PER; t++) {
        const double mt = (AX < D - 1) ? m0 : M[row[t] * (NC + 1) + mm];
        const double bt = (AX == D - 1 && N > NT) ? b0 : buf[line[t] + mm * st];
        out[t] = out[t] + mt * bt;
      }
    }
  }
  __syncthreads();
  if (tid < N)
#pragma unroll
    for (int t = 0; t < PER; t++) buf[tid + t * NT] = out[t];
  __syncthreads();
}
// The level-1 solve on buf (interior cells, x fastest): V^-1 along each
// axis, division by the eigenvalue sums, V along each axis.  mat: the 2 D
// matrices, V^-1 first, rows padded to NC + 1.
template <int D, int NC, int NT>
__device__ inline void coarse_transforms(double *buf, const double *mat, const double *__restrict__ eig,
                                         double lambda2) {
  constexpr int MS = NC * (NC + 1);
  coarse_axis<D, NC, NT, 0>(buf, mat);
  coarse_axis<D, NC, NT, 1>(buf, mat + MS);
  if constexpr (D == 3) coarse_axis<D, NC, NT, 2>(buf, mat + 2 * MS);
  for (int q = threadIdx.x; q < Geo<D, NC>::NINT; q += NT) {
    int i, j, k;
    interior_ijk<D, NC>(q, i, j, k);
    double den = eig[i - 1] + eig[NC + j - 1];
    if (D == 3) den = den + eig[2 * NC + k - 1];
    den = den - lambda2;
    buf[q] = buf[q] / den;
  }
  __syncthreads();
  coarse_axis<D, NC, NT, 0>(buf, mat + D * MS);
  coarse_axis<D, NC, NT, 1>(buf, mat + (D + 1) * MS);
  if constexpr (D == 3) coarse_axis<D, NC, NT, 2>(buf, mat + (D + 2) * MS);
}

// Exact level-1 solve by fast diagonalisation (replaces hypre PFMG,
// afivo/src/m_coarse_solver.f90:421): fold boundary values into the rhs,
// transform with V^-1 along each axis, divide by the eigenvalue sums,
// transform back with V.  One workgroup of CBS threads per level-1 box (one
// per run of a forest); the box and the matrices live in LDS.  Bound by the
// 2 D dependent products of one workgroup: 17 us for a 16^3 box, and 52 us
// with the matrices read from memory by every cell.
// TS is the storage type of rhs and phi; the transforms always run in FP64.
template <int D, int NC, int CBS, typename TS>
__global__ void __launch_bounds__(CBS) k_coarse_solve(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                      const TS *rhs,
                                                      TS *phi, VarBc m, double lambda2, int cyl,
                                                      const double *__restrict__ vinv,
                                                      const double *__restrict__ v,
                                                      const double *__restrict__ eig) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, TS>;
  constexpr int N = G::NINT;
  __shared__ double buf[N];
  __shared__ double mat[2 * D * NC * (NC + 1)];
  const int id = ids[blockIdx.x];
  if (id <= 0) return;  // run masked out
  const DBox &bx = boxes[id - 1];
  const Sten<D, double> s = lpl_stencil<D, double>(bx, lambda2);
  const TS *r = rhs + (size_t)(id - 1) * L::STRIDE;
  for (int q = threadIdx.x; q < 2 * D * NC * NC; q += CBS)
    mat[(q / NC) * (NC + 1) + q % NC] = (q < D * NC * NC) ? vinv[q] : v[q - D * NC * NC];
  for (int q = threadIdx.x; q < N; q += CBS) {
    int i, j, k;
    interior_ijk<D, NC>(q, i, j, k);
    buf[q] = coarse_rhs_value<D, NC>(bx, m, s, cyl != 0, (double)r[L::in_at(i, j, k)], i, j, k);
  }
  __syncthreads();
  coarse_transforms<D, NC, CBS>(buf, mat, eig, lambda2);
  TS *u = phi + (size_t)(id - 1) * L::STRIDE;
  for (int q = threadIdx.x; q < N; q += CBS) {
    int i, j, k;
    interior_ijk<D, NC>(q, i, j, k);
    u[L::in_at(i, j, k)] = (TS)buf[q];
  }
}

// ---- mixed precision: the FP64 side of the defect correction ---------------
// The inner multigrid cycle works on the correction e (single precision,
// homogeneous boundary conditions) of the FP64 potential; these two kernels
// close each cycle in FP64.

// FP64 residual rhs - L phi on the interior cells of a box list, with every
// neighbour outside the box taken from ghost_value() (so the stored ghost
// layer of phi need not be current), stored in single precision as the rhs
// of the next correction cycle; max |residual| over leaf boxes is reduced
// into *leafmax.
template <int D, int NC, int BS, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_mp_residual(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                         const double *__restrict__ phi, const double *__restrict__ rhs,
                                                         float *r32, double lambda2, int cyl, VarBc m,
                                                         unsigned long long *leafmax, int bpb, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, float>;
  __shared__ double sh[BS / 64];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const Part pt = part_of<BS>(ids, bpb, w);
    if (pt.id <= 0) continue;  // run masked out
    const int id = pt.id;
    const DBox &bx = boxes[id - 1];
    const Sten<D, double> s = lpl_stencil<D, double>(bx, lambda2);
    const size_t base = (size_t)(id - 1) * G::NCELL;
    const double *u = phi + base;
    float *r = r32 + (size_t)(id - 1) * L::STRIDE;
    constexpr int st[3] = {1, G::NG, G::NG * G::NG};
    double mx = 0;
    for (int q = pt.q0; q < G::NINT; q += pt.stride) {
      int i, j, k;
      interior_ijk<D, NC>(q, i, j, k);
      const int x = G::idx(i, j, k);
      const int pos[3] = {i, j, k};
      const double uc = u[x];
      double nbv[6];
      for (int nb = 0; nb < 2 * D; nb++) {
        const int d = nb / 2;
        const bool low = (nb % 2) == 0;
        const bool edge = low ? pos[d] == 1 : pos[d] == NC;
        if (!edge) {
          nbv[nb] = u[low ? x - st[d] : x + st[d]];
        } else {
          int t0, t1;
          tangential(D, d, t0, t1);
          const double x2 = u[low ? x + st[d] : x - st[d]];
          nbv[nb] = ghost_value<D, NC, double>(boxes, bx, phi, m, nb, pos[t0], (D == 3) ? pos[t1] : 0, uc, x2);
        }
      }
      double lp;
      if (D == 2) {
        if (cyl) {
          double c1, c2, c3;
          cyl_coeffs<double>(bx, i, s.c, c1, c2, c3);
          lp = c1 * uc + c2 * nbv[0] + c3 * nbv[1] + s.c[3] * nbv[2] + s.c[4] * nbv[3];
        } else {
          lp = s.c[0] * uc + s.c[1] * nbv[0] + s.c[2] * nbv[1] + s.c[3] * nbv[2] + s.c[4] * nbv[3];
        }
      } else {
        lp = s.c[0] * uc + s.c[1] * nbv[0] + s.c[2] * nbv[1] + s.c[3] * nbv[2] + s.c[4] * nbv[3] +
             s.c[5] * nbv[4] + s.c[6] * nbv[5];
      }
      const double rv = rhs[base + x] - lp;
      r[L::in_at(i, j, k)] = (float)rv;
      mx = fmax(mx, fabs(rv));
    }
    if (bx.children[0] == 0) {
      mx = group_max<BS, BB>(mx, sh);
      if (ltid<BS>() == 0) atomic_max_nonneg(run_slot(leafmax, bx), mx);
    }
  }
}

// ---- LDS-staged forms (one workgroup per box) ---------------------------------
// The box interior is loaded once, coalesced, into LDS with the face ghosts
// that the pass needs (Stage: copied from the neighbours, or formed by
// staged_ghost, ghost_value's operations); the stencil then reads LDS only.
// k_smooth_block forms its ghosts by ghost_value itself.

template <int D, int NC, int BS, typename T, int BB = 1>
__device__ inline void lds_load_interior(T *s, const T *u) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  for (int q = ltid<BS>(); q < G::NINT; q += BS) {
    int i, j, k;
    interior_ijk<D, NC>(q, i, j, k);
    s[G::idx(i, j, k)] = u[L::in_at(i, j, k)];
  }
}

// v[n] for a small n that differs between lanes, without indexed registers
// or a load per lane (v: kernel arguments, a box record's uniform fields).
// (The values are selected, not their addresses: a selected address keeps
// the whole array in scratch memory.)
template <int N, typename V>
__device__ inline V pick(const V *v, int n) {
  if constexpr (N == 1) {
    return V(v[0]);
  } else {
    const V lower = pick<N - 1>(v, n), last = V(v[N - 1]);
    return (n == N - 1) ? V(last) : V(lower);
  }
}
// Cell (i, j, k) at normal index pn and tangential (a, b) of face nb, for an
// nb that may differ between lanes.
template <int D>
__device__ inline void face_cell(int nb, int a, int b, int pn, int &i, int &j, int &k) {
  const int d = nb >> 1;
  i = (d == 0) ? pn : a;
  j = (d == 1) ? pn : (D == 2 || d == 0) ? a : b;
  k = (D == 2) ? 0 : (d == 2) ? pn : b;
}
// The coarse cells the ghosts of a face at a refinement boundary are formed
// from: the face layer of the coarse neighbour over the box's extent and one
// cell around it.  Patch cell pa (+ PP pb) holds the coarse cell at
// tangential (co[t0] + pa, co[t1] + pb), co the box's offset within its
// parent.
template <int D, int NC>
struct CoarsePatch {
  static constexpr int PP = NC / 2 + 2;
  static constexpr int N = (D == 3) ? PP * PP : PP;
};
// The coarse values ghost_coarse_load reads for ghost (a, b)
// (mg_sides_rb, afivo/src/m_af_multigrid.f90:294-461; af_gc_interp(_lim),
// afivo/src/m_af_ghostcell.f90:394-605), in its order, from the patch.
template <int D, int NC, typename T>
__device__ inline CoarseVals<T> coarse_patch_vals(const T *cp, const VarBc &m, int a, int b) {
  constexpr int PP = CoarsePatch<D, NC>::PP;
  auto at = [&](int qa, int qb) { return cp[D == 3 ? qa + PP * qb : qa]; };
  CoarseVals<T> cv = {{T(0), T(0), T(0), T(0), T(0)}};
  if (m.rb == RB_MG) {
    const int i = (a + 1) >> 1, j = (b + 1) >> 1;
    cv.v[0] = at(i + 1, j);
    cv.v[1] = at(i - 1, j);
    if (D == 2) {
      cv.v[2] = at(i, j);
    } else {
      cv.v[2] = at(i, j + 1);
      cv.v[3] = at(i, j - 1);
      cv.v[4] = at(i, j);
    }
    return cv;
  }
  const int a1 = (a + 1) >> 1, a2 = a1 + 1 - 2 * (a & 1);
  const int b1 = (b + 1) >> 1, b2 = b1 + 1 - 2 * (b & 1);
  cv.v[0] = at(a1, b1);
  cv.v[1] = at(a2, b1);
  if (D == 3) cv.v[2] = at(a1, b2);
  return cv;
}
// Ghost of a face on the physical boundary from the box's first and second
// cells x1, x2: p + c1 x1 + 0 x2 (ghost_value's operations, for an nb that
// may differ between lanes).  dr: the box's spacing; run_val: the run's value
// of face m.run_face.
template <int D, typename T>
__device__ inline void phys_coeffs(const double *dr, const VarBc &m, double run_val, int nb, T &p, T &c1) {
  const int type = pick<2 * D>(m.type, nb);
  const double bv = (m.run_val && nb == m.run_face) ? run_val : pick<2 * D>(m.val, nb);
  T c0;
  if (type == BC_DIRICHLET) {
    c0 = 2;
    c1 = -1;
  } else if (type == BC_NEUMANN) {
    c0 = (T)pick<D>(dr, nb >> 1) * T((nb & 1) ? 1 : -1);
    c1 = 1;
  } else {
    c0 = 1;
    c1 = 0;
  }
  p = c0 * (T)bv;
}
template <int D, typename T>
__device__ inline T phys_ghost(const DBox &bx, const VarBc &m, double run_val, int nb, T x1, T x2) {
  T p, c1;
  phys_coeffs<D, T>(bx.dr, m, run_val, nb, p, c1);
  return p + c1 * x1 + T(0) * x2;
}
// Ghost (a, b) of a face without a same-level neighbour (nbv <= 0) from the
// box's first and second cells x1, x2 and, at a refinement boundary, the
// face's coarse patch cp.
template <int D, int NC, typename T>
__device__ inline T staged_ghost(const DBox &bx, const VarBc &m, double run_val, int nbv, int nb, int a, int b,
                                 const T *cp, T x1, T x2) {
  if (nbv < 0) return phys_ghost<D, T>(bx, m, run_val, nb, x1, x2);
  const CoarseVals<T> cv = coarse_patch_vals<D, NC, T>(cp, m, a, b);
  const GhostPart<T> g = coarse_part<D, T>(m, nb >> 1, a, b, cv);
  return rb_finish<T>(m, g, x1, x2);
}

// Staging of a box and its face ghosts into LDS in one memory round.  The
// box record's fields are uniform; every lane issues its loads without
// branches (the interior, and per face ghost one value: the same-level
// neighbour's cell across the face, which is the ghost, or the box's own
// first cell; then, in boxes at a refinement boundary, the coarse patches of
// the faces there), so all of them are in flight together.  After a barrier
// the ghosts of the faces without a neighbour are formed from LDS.  What
// bounds it is that chain, record -> cells -> LDS, not the bytes, on all but
// the largest levels.  A form with a branch per ghost and indexed face
// fields waited for its loads branch by branch and kept the boundary methods
// in scratch memory: per launch, the half-sweep of a refined mesh of 8^2
// FP64 boxes then took 10.1 us (now 3.2), of 4000 8^3 FP32 boxes 21.7 us
// (8.2), of 16^3 FP64 boxes 16.8 us (13.8); the FP64 residual of 1024 8^2
// boxes 17.5 us (3.9), of 1856 16^3 boxes 45.1 us (41.6).
// COL: only the ghosts next to interior cells of GSRB colour `colour`, and
// in the colour-split FP32 layout only the interior cells of the other
// colour, the only ones a half-sweep of that colour reads.
// stored: the face ghosts are the box's own stored ghost layer (the
// reference's smoother reads that layer as it stands before its first
// half-sweep; FP64 layout only).
// issue() makes the loads, commit() the LDS copy s (afivo's order), with cp
// (2 D CoarsePatch::N values) as scratch, and ends with a barrier; between
// the two a kernel can do work that needs neither.
template <int D, int NC, int BS, typename T, int BB, bool COL>
struct Stage {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  using P = CoarsePatch<D, NC>;
  static constexpr bool ONE = L::SPLIT && COL;
  static constexpr int NL = ONE ? G::NINT / 2 : G::NINT;  // interior cells loaded
  static constexpr int NI = (NL + BS - 1) / BS;
  static constexpr int NE = COL ? G::NTAN / 2 : G::NTAN;  // ghosts of a face
  static constexpr int NGH = 2 * D * NE, NF = (NGH + BS - 1) / BS;
  static constexpr int NPT = 2 * D * P::N, NP = (NPT + BS - 1) / BS;
  T vi[NI], vf[NF], vp[NP];
  int nbid[2 * D];
  int colour;
  bool any_rb, any_b, stored;
  double run_val;

  // interior cell (i, j, k) of load q and its position in the pool: in the
  // split layout the loads run over the colour blocks in order
  __device__ int cell(int q, int &i, int &j, int &k) const {
    if constexpr (L::SPLIT) {
      constexpr int HALF = G::NINT / 2;
      const int x = q + (ONE ? (1 - colour) * HALF : 0);
      colour_cell<D, NC>(x >= HALF, x >= HALF ? x - HALF : x, i, j, k);
      return x;
    } else {
      interior_ijk<D, NC>(q, i, j, k);
      return L::in_at(i, j, k);
    }
  }
  // ghost item q: its face and tangential position (COL: next to a cell
  // with (i + j + k + colour) even)
  __device__ void item(int q, int &nb, int &a, int &b) const {
    nb = q / NE;
    const int e = q % NE;
    if constexpr (COL) {
      const int pd = (nb & 1) ? NC : 1;
      b = (D == 3) ? e / (NC / 2) + 1 : 0;
      a = 2 * (e % (NC / 2)) + 1 + ((colour + pd + b + 1) & 1);
    } else {
      a = e % NC + 1;
      b = (D == 3) ? e / NC + 1 : 0;
    }
  }

  __device__ void issue(const DBox &bx, int id, const T *var, const VarBc &m, int colour_, const T *coarse = nullptr,
                        bool stored_ = false) {
    colour = colour_;
    stored = stored_ && !L::SPLIT;
    any_rb = any_b = false;
#pragma unroll
    for (int nb = 0; nb < 2 * D; nb++) {
      nbid[nb] = __builtin_amdgcn_readfirstlane(bx.nb[nb]);
      any_b = any_b || nbid[nb] <= 0;
      any_rb = any_rb || nbid[nb] == 0;
    }
    any_b = any_b && !stored;
    any_rb = any_rb && !stored;
    const T *u = var + (size_t)(id - 1) * L::STRIDE;
#pragma unroll
    for (int t = 0; t < NI; t++) {
      int q = ltid<BS>() + t * BS;
      if (NL % BS) q = min(q, NL - 1);
      int i, j, k;
      vi[t] = u[cell(q, i, j, k)];
    }
#pragma unroll
    for (int t = 0; t < NF; t++) {
      int q = ltid<BS>() + t * BS;
      if (NGH % BS) q = min(q, NGH - 1);
      int nb, a, b, i, j, k;
      item(q, nb, a, b);
      const int nbv = pick<2 * D>(nbid, nb);
      const bool low = (nb & 1) == 0, copy = nbv > 0 && !stored;
      const int pn = stored ? (low ? 0 : NC + 1) : (copy == low) ? NC : 1;
      face_cell<D>(nb, a, b, pn, i, j, k);
      const T *from = var + (size_t)((copy ? nbv : id) - 1) * L::STRIDE;
      vf[t] = from[L::SPLIT ? L::in_at(i, j, k) : L::at(i, j, k)];
    }
    if (any_rb) {
      const T *cvar = coarse ? coarse : var;
      int co[3];
#pragma unroll
      for (int d = 0; d < D; d++) co[d] = ((bx.ix[d] - 1) & 1) * (NC / 2);
#pragma unroll
      for (int t = 0; t < NP; t++) {
        const int q = min(ltid<BS>() + t * BS, NPT - 1);
        const int nb = q / P::N, e = q % P::N, d = nb >> 1;
        const bool rb = pick<2 * D>(nbid, nb) == 0;
        const int c0 = (d == 0) ? co[1] : co[0], c1 = (D == 2) ? 0 : (d == 2) ? co[1] : co[2];
        int i, j, k;
        face_cell<D>(nb, c0 + e % P::PP, (D == 3) ? c1 + e / P::PP : 0, (nb & 1) ? 1 : NC, i, j, k);
        const T *from = rb ? cvar + (size_t)(pick<2 * D>(bx.pnb, nb) - 1) * L::STRIDE + L::at(i, j, k) : u;
        vp[t] = *from;
      }
    }
    run_val = (any_b && m.run_val) ? m.run_val[bx.run] : 0.0;
  }

  __device__ void commit(T *s, T *cp, const DBox &bx, const VarBc &m) {
#pragma unroll
    for (int t = 0; t < NI; t++) {
      const int q = ltid<BS>() + t * BS;
      int i, j, k;
      cell(q, i, j, k);
      if (NL % BS == 0 || q < NL) s[G::idx(i, j, k)] = vi[t];
    }
#pragma unroll
    for (int t = 0; t < NF; t++) {
      const int q = ltid<BS>() + t * BS;
      if (NGH % BS && q >= NGH) continue;
      int nb, a, b, i, j, k;
      item(q, nb, a, b);
      face_cell<D>(nb, a, b, (nb & 1) ? NC + 1 : 0, i, j, k);
      // (the ghosts of the other faces are written again below)
      s[G::idx(i, j, k)] = vf[t];
    }
    if (any_rb) {
#pragma unroll
      for (int t = 0; t < NP; t++) {
        const int q = ltid<BS>() + t * BS;
        if (q < NPT) cp[q] = vp[t];
      }
    }
    gsync<BS, BB>();
    if (!any_b) return;
#pragma unroll
    for (int t = 0; t < NF; t++) {
      const int q = ltid<BS>() + t * BS;
      if (NGH % BS && q >= NGH) continue;
      int nb, a, b, i, j, k;
      item(q, nb, a, b);
      const int nbv = pick<2 * D>(nbid, nb);
      if (nbv > 0) continue;
      face_cell<D>(nb, a, b, (nb & 1) ? NC - 1 : 2, i, j, k);
      const T x2 = s[G::idx(i, j, k)];
      face_cell<D>(nb, a, b, (nb & 1) ? NC + 1 : 0, i, j, k);
      s[G::idx(i, j, k)] = staged_ghost<D, NC, T>(bx, m, run_val, nbv, nb, a, b, cp + nb * P::N, vf[t], x2);
    }
    gsync<BS, BB>();
  }
};

// Red-black Gauss-Seidel half-sweep (stencil_gsrb_357,
// m_af_stencil.f90:838-998) fused with the ghost-cell fill that the
// reference performs before it (gsrb_boxes, m_af_multigrid.f90:648-687):
// a neighbour outside the box is taken from ghost_value() with the same
// inputs af_gc_box would use, so the updated cells are bit-identical while
// no separate ghost-fill pass is needed between half-sweeps.  (The stored
// ghost layer is refreshed once after the last half-sweep.)  stored: the
// first half-sweep of a V-cycle's finest level reads the stored layer as
// the reference does, also where it is out of date (the neighbours of boxes
// just added or removed by refinement).
// One workgroup (or, for 8^2 boxes, wavefront) per box, the box in LDS.
template <int D, int NC, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_gsrb_lds(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                      T *phi, const T *__restrict__ rhs, int redblack, T lambda2,
                                                      int cyl, VarBc m, int stored, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  __shared__ T s_all[BB][G::NCELL];
  __shared__ T cp_all[BB][2 * D * CoarsePatch<D, NC>::N];
  T *s = s_all[lgrp<BS, BB>()], *cp = cp_all[lgrp<BS, BB>()];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const int id = __builtin_amdgcn_readfirstlane(ids[w]);
    if (id <= 0) continue;  // run masked out
    const DBox &bx = boxes[id - 1];
    T *u = phi + (size_t)(id - 1) * L::STRIDE;
    const T *r = rhs + (size_t)(id - 1) * L::STRIDE;
    constexpr int HALF = G::NINT / 2;
    constexpr int NH = (HALF + BS - 1) / BS;
    constexpr int sx = 1, sy = G::NG, sz = G::NG * G::NG;
    // updated cell t of this thread, and its rhs (loaded with the box)
    auto cell = [&](int q, int &i, int &j, int &k) {
      const int mm = q % (NC / 2);
      j = (q / (NC / 2)) % NC + 1;
      k = (D == 3) ? q / ((NC / 2) * NC) + 1 : 0;
      const int i0 = 2 - ((redblack ^ (D == 3 ? k + j : j)) & 1);
      i = i0 + 2 * mm;
    };
    T rr[NH];
    for (int t = 0; t < NH; t++) {
      const int q = ltid<BS>() + t * BS;
      if (q < HALF) {
        int i, j, k;
        cell(q, i, j, k);
        rr[t] = r[L::SPLIT ? (redblack & 1) * HALF + q : L::in_at(i, j, k)];
      }
    }
    // the updated cells satisfy (i + j + k + redblack) even
    Stage<D, NC, BS, T, BB, true> sg;
    sg.issue(bx, id, phi, m, redblack & 1, nullptr, stored != 0);
    const Sten<D, T> st = lpl_stencil<D, T>(bx, lambda2);
    sg.commit(s, cp, bx, m);
    for (int t = 0; t < NH; t++) {
      const int q = ltid<BS>() + t * BS;
      if (q >= HALF) break;
      int i, j, k;
      cell(q, i, j, k);
      const int x = G::idx(i, j, k);
      const T rx = rr[t];
      if (D == 2) {
        if (cyl) {
          T c1, c2, c3;
          cyl_coeffs<T>(bx, i, st.c, c1, c2, c3);
          T inv1 = T(1) / c1;
          s[x] = (rx - c2 * s[x - sx] - c3 * s[x + sx] - st.c[3] * s[x - sy] - st.c[4] * s[x + sy]) * inv1;
        } else {
          T inv_c1 = T(1) / st.c[0];
          s[x] = (rx - st.c[1] * s[x - sx] - st.c[2] * s[x + sx] - st.c[3] * s[x - sy] - st.c[4] * s[x + sy]) *
                 inv_c1;
        }
      } else {
        T inv_c1 = T(1) / st.c[0];
        s[x] = (rx - st.c[1] * s[x - sx] - st.c[2] * s[x + sx] - st.c[3] * s[x - sy] - st.c[4] * s[x + sy] -
                st.c[5] * s[x - sz] - st.c[6] * s[x + sz]) *
               inv_c1;
      }
    }
    gsync<BS, BB>();
    if (L::SPLIT) {
      // the updated colour's block
      for (int q = ltid<BS>(); q < HALF; q += BS) {
        int i, j, k;
        cell(q, i, j, k);
        u[(redblack & 1) * HALF + q] = s[G::idx(i, j, k)];
      }
    } else {
      // Whole interior rows back (the other colour unchanged): full-line
      // stores instead of every other word, so no line has to be fetched to
      // merge a partial write.  Neighbouring boxes only read this box's
      // other colour during the launch, which keeps its value.
      for (int q = ltid<BS>(); q < G::NINT; q += BS) {
        int i, j, k;
        interior_ijk<D, NC>(q, i, j, k);
        const int x = G::idx(i, j, k);
        u[x] = s[x];
      }
    }
    gsync<BS, BB>();  // (the group's LDS is reused by its next item)
  }
}

// k_gsrb_lds for 3D boxes in the colour-split single-precision layout.  A
// half-sweep reads only the other colour's interior, the face ghosts next to
// the updated cells and the updated colour's rhs; the updated colour's old
// values are never read (but for the cells next to faces without a
// same-level neighbour, whose ghosts use them).  Everything a box reads goes
// straight from memory into LDS (global_load_lds, no registers held): the
// other colour's block and the rhs as they lie in the pool (16-byte words),
// and for each face either the same-level neighbour's cells across it (one
// value per ghost, already the ghost) or the box's own cells next to it and,
// at a refinement boundary, a patch of the coarse neighbour's face layer.
// After one barrier those faces' ghosts are formed, after a second each
// thread updates four consecutive cells of the colour block per pass and
// stores them as one 16-byte word.  The stencil and ghost expressions and
// their operands are those of k_gsrb_lds, so the results are identical.
// With few registers and 25 KB of LDS, six boxes fit on a CU: all 1536
// boxes of a 256-CU finest level run at once.
constexpr int GSRB_SPLIT_NT = 256;
template <int D, int NC, int NT>
__global__ void __launch_bounds__(NT) k_gsrb_split(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                   float *phi, const float *__restrict__ rhs, int redblack,
                                                   float lambda2, VarBc m, int nw) {
  static_assert(D == 3, "the colour blocks of 3D boxes");
  using G = Geo<D, NC>;
  using L = Lay<D, NC, float>;
  constexpr int HALF = L::HALF;
  constexpr int NV = HALF / 4;               // 16-byte words of a colour block
  constexpr int NW = NV / NT;                // per thread
  constexpr int NE = G::NTAN / 2;            // ghosts of a face next to updated cells
  constexpr int NGH = 2 * D * NE;            // of the box
  constexpr int NGT = (NGH + NT - 1) / NT;   // per thread
  constexpr int PP = NC / 2 + 2;             // coarse patch of a face: its coarse cells and a ring
  static_assert(NV % NT == 0 && (L::STRIDE * sizeof(float)) % 16 == 0, "16-byte words of whole boxes");
  static_assert(NE % 64 == 0 && NT % 64 == 0 && PP * PP <= NE, "a face's ghosts in whole wavefronts");
  __shared__ float4 s_other4[NV];
  __shared__ float4 s_rhs4[NV];
  __shared__ float s_gh[2 * D][NE];  // the ghosts: face nb, item e
  __shared__ float s_x1[2 * D][NE];  // the box's cells next to a face without a same-level neighbour
  __shared__ float s_cp[2 * D][NE];  // the coarse patch of a face at a refinement boundary
  const float *s_other = reinterpret_cast<const float *>(s_other4);
  const int t = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(t / 64);  // (the wavefront)
  const int uc = redblack & 1, oc = 1 - uc;  // updated cells: (i + j + k + redblack) even
  // ghost item e of face nb: tangential (a, b), next to an updated cell
  auto item_ab = [&](int nb, int e, int &a, int &b) {
    const int pd = (nb % 2) == 0 ? 1 : NC;
    b = e / (NC / 2) + 1;
    a = 2 * (e % (NC / 2)) + 1 + ((uc + pd + b + 1) & 1);  // (pd + a + b + uc) even
  };
  for (int w = blockIdx.x; w < nw; w += gridDim.x) {
    const int id = ids[w];
    if (id <= 0) continue;  // run masked out
    const DBox &bx = boxes[id - 1];
    const Sten<D, float> st = lpl_stencil<D, float>(bx, lambda2);
    float *u = phi + (size_t)(id - 1) * L::STRIDE;
    const float4 *ob = reinterpret_cast<const float4 *>(u + oc * HALF);
    const float4 *rb = reinterpret_cast<const float4 *>(rhs + (size_t)(id - 1) * L::STRIDE + uc * HALF);
    for (int q = 0; q < NW; q++) {
      __builtin_amdgcn_global_load_lds((const void *)(ob + t + q * NT),
                                       (__attribute__((address_space(3))) void *)(s_other4 + 64 * wv + q * NT), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void *)(rb + t + q * NT),
                                       (__attribute__((address_space(3))) void *)(s_rhs4 + 64 * wv + q * NT), 16, 0, 0);
    }
    int nbid[2 * D];
    for (int nb = 0; nb < 2 * D; nb++) nbid[nb] = bx.nb[nb];
    // the faces' values, one per lane: a wavefront's items lie on one face
    // (its face, its first item and the neighbour there are uniform), and
    // item e of a wavefront lands at e of the face's arrays
    for (int q = 0; q < NGT; q++) {
      const int g0 = 64 * wv + q * NT;
      if (g0 >= NGH) continue;
      const int nb = g0 / NE, e0 = g0 % NE, e = e0 + (t & 63);
      const int nbv = __builtin_amdgcn_readfirstlane(nbid[nb]);
      const bool low = (nb % 2) == 0;
      int a, b, p[3];
      item_ab(nb, e, a, b);
      if (nbv > 0) {  // the same-level neighbour's cell across the face: the ghost
        face_pos<D>(nb, a, b, low ? NC : 1, p);
        const float *src = phi + (size_t)(nbv - 1) * L::STRIDE + L::in_at(p[0], p[1], p[2]);
        __builtin_amdgcn_global_load_lds((const void *)src, (__attribute__((address_space(3))) void *)&s_gh[nb][e0],
                                         4, 0, 0);
      } else {
        face_pos<D>(nb, a, b, low ? 1 : NC, p);
        __builtin_amdgcn_global_load_lds((const void *)(u + L::in_at(p[0], p[1], p[2])),
                                         (__attribute__((address_space(3))) void *)&s_x1[nb][e0], 4, 0, 0);
        if (nbv == 0 && e < PP * PP) {  // refinement boundary: coarse patch cell e
          const int d = nb / 2;
          int t0, t1;
          tangential(D, d, t0, t1);
          int qc[3];
          qc[d] = low ? NC : 1;
          qc[t0] = ((bx.ix[t0] - 1) & 1) * (NC / 2) + e % PP;
          qc[t1] = ((bx.ix[t1] - 1) & 1) * (NC / 2) + e / PP;
          const float *P = phi + (size_t)(__builtin_amdgcn_readfirstlane(bx.pnb[nb]) - 1) * L::STRIDE;
          __builtin_amdgcn_global_load_lds((const void *)(P + L::at(qc[0], qc[1], qc[2])),
                                           (__attribute__((address_space(3))) void *)&s_cp[nb][e0], 4, 0, 0);
        }
      }
    }
    __syncthreads();
    // the ghosts of faces without a same-level neighbour (the box's second
    // cell along the normal is of the other colour: in the staged block)
    for (int q = 0; q < NGT; q++) {
      const int g0 = 64 * wv + q * NT;
      if (g0 >= NGH) continue;
      const int nb = g0 / NE, e = g0 % NE + (t & 63);
      const int nbv = __builtin_amdgcn_readfirstlane(nbid[nb]);
      if (nbv > 0) continue;
      const bool low = (nb % 2) == 0;
      int a, b, p[3];
      item_ab(nb, e, a, b);
      face_pos<D>(nb, a, b, low ? 2 : NC - 1, p);
      const float x2 = s_other[L::in_at(p[0], p[1], p[2]) - oc * HALF];
      CoarseVals<float> cv = {{0.0f, 0.0f, 0.0f, 0.0f, 0.0f}};
      if (nbv == 0) cv = coarse_patch_vals<D, NC, float>(s_cp[nb], m, a, b);
      s_gh[nb][e] =
          ghost_finish<D, NC, float>(bx, m, nb, ghost_coarse_form<D, NC, float>(bx, m, nb, a, b, cv), s_x1[nb][e], x2);
    }
    __syncthreads();
    const float inv_c1 = 1.0f / st.c[0];
    float4 *ub = reinterpret_cast<float4 *>(u + uc * HALF);
    for (int q = 0; q < NW; q++) {
      // four cells: half of a row (j, k) of the colour block, at
      // i = i0 + 2 (m0 + c); their other-colour neighbours in the row are
      // the five values from B on, in the rows and planes beside it four
      // consecutive values (one 16-byte word), unless they are ghosts
      const int h0 = 4 * (t + q * NT);
      const int row = h0 / (NC / 2), m0 = h0 % (NC / 2);
      const int j = row % NC + 1, k = row / NC + 1;
      const int i0 = 1 + ((1 + j + k + uc) & 1);
      const int R = row * (NC / 2);
      const int B = R + m0 + i0 - 2;
      // (one 16-byte word at R + m0 and one value before or after it:
      // consecutive lanes read consecutive words, free of bank conflicts)
      const bool lo_gh = i0 == 1 && m0 == 0, hi_gh = i0 == 2 && m0 == NC / 2 - 4;
      const float4 xc = s_other4[(R + m0) / 4];
      // (a face's ghosts are stored every other cell: cell r of the face
      // at r / 2)
      const float xe = (i0 == 1) ? (lo_gh ? s_gh[0][row >> 1] : s_other[max(B, 0)])
                                 : (hi_gh ? s_gh[1][row >> 1] : s_other[min(B + 4, HALF - 1)]);
      float xw[5];
      if (i0 == 1) {
        xw[0] = xe; xw[1] = xc.x; xw[2] = xc.y; xw[3] = xc.z; xw[4] = xc.w;
      } else {
        xw[0] = xc.x; xw[1] = xc.y; xw[2] = xc.z; xw[3] = xc.w; xw[4] = xe;
      }
      float ym[4], yp[4], zm[4], zp[4];
      auto four = [&](float *v, bool ghost, int nb, int r0, int off) {
        if (ghost) {
          for (int c = 0; c < 4; c++) v[c] = s_gh[nb][(r0 + i0 - 1 + 2 * (m0 + c)) >> 1];
        } else {
          const float4 w = s_other4[min(max(R + off + m0, 0), HALF - 4) / 4];
          v[0] = w.x;
          v[1] = w.y;
          v[2] = w.z;
          v[3] = w.w;
        }
      };
      four(ym, j == 1, 2, NC * (k - 1), -NC / 2);
      four(yp, j == NC, 3, NC * (k - 1), NC / 2);
      four(zm, k == 1, 4, NC * (j - 1), -NC * NC / 2);
      four(zp, k == NC, 5, NC * (j - 1), NC * NC / 2);
      const float4 rv = s_rhs4[t + q * NT];
      const float rr[4] = {rv.x, rv.y, rv.z, rv.w};
      float res[4];
      for (int c = 0; c < 4; c++)
        res[c] = (rr[c] - st.c[1] * xw[c] - st.c[2] * xw[c + 1] - st.c[3] * ym[c] - st.c[4] * yp[c] -
                  st.c[5] * zm[c] - st.c[6] * zp[c]) *
                 inv_c1;
      ub[t + q * NT] = make_float4(res[0], res[1], res[2], res[3]);
    }
    __syncthreads();  // (the LDS is reused by the next item)
  }
}

// k_gsrb_lds for 2D boxes of 8^2 cells in the colour-split single-precision
// layout (the ensembles' half-sweep).  A wavefront takes eight boxes, a lane
// one row of the box's updated colour (four cells, one 16-byte word).  All
// that the eight boxes read goes straight from memory into the wavefront's
// part of LDS (global_load_lds, one round, no registers held): each row's
// other-colour word and rhs word, the row's x ghost (the neighbour's cell
// across the face), the y ghosts (the neighbour's facing row of the other
// colour, one word per face), and for a face without a same-level neighbour
// the box's own cells next to it and the coarse values its ghosts need.
// Those ghosts are then formed in LDS, and each lane updates its row.  The
// ghost and stencil expressions and their operands are those of
// k_gsrb_lds, so the results are identical.  Wavefronts never wait for
// each other.
#define LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))
template <int NC>
__global__ void __launch_bounds__(256) k_gsrb_split2d(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                      float *phi, const float *__restrict__ rhs, int redblack,
                                                      float lambda2, int cyl, VarBc m, int n_boxes, int nw) {
  constexpr int D = 2;
  using L = Lay<D, NC, float>;
  constexpr int HALF = L::HALF;
  static_assert(NC == 8 && HALF == 32 && (L::STRIDE * sizeof(float)) % 16 == 0, "8^2 boxes: a row is one word");
  constexpr int NBW = 8;                       // boxes per wavefront
  __shared__ float4 s_o[4][64];                // other colour, row r of box bl at lane 8 bl + r
  __shared__ float4 s_r[4][64];                // rhs of the updated colour, the same
  __shared__ float4 s_y[4][64];                // y ghosts of box bl: face 2 at 8 bl, face 3 at 8 bl + 4
  __shared__ float s_gx[4][64];                // x ghost of row r
  __shared__ float s_x1[2][4][64];             // the box's cell next to a face: x item, y item
  __shared__ float s_cv[2][3][4][64];          // coarse values of an item at a refinement boundary
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x & 63;
  const int bl = lane >> 3, r = lane & 7;
  const int uc = redblack & 1, oc = 1 - uc;    // updated cells: (i + j + redblack) even
  for (int w = xcd_item(); w < nw; w += gridDim.x) {
    const int b = (4 * w + wv) * NBW + bl;
    const int id = b < n_boxes ? ids[b] : 0;
    const bool on = id > 0;  // (past the end, or a run masked out)
    const DBox &bx = boxes[on ? id - 1 : 0];
    float *u = phi + (size_t)(on ? id - 1 : 0) * L::STRIDE;
    const int j = r + 1, i0 = 1 + ((1 + j + uc) & 1);
    // x item: the ghost of row j on the side of its first or last cell
    const int nbx = (i0 == 1) ? 0 : 1;
    // y item: face 2 (r < 4) or 3, the cell i = i0y + 2 mm of the face row
    const int fy = r >> 2, mm = r & 3, nby = 2 + fy, jy = fy ? NC : 1;
    const int iy = 1 + ((1 + jy + uc) & 1) + 2 * mm;
    int nbvx = 0, nbvy = 0;
    if (on) {
      nbvx = bx.nb[nbx];
      nbvy = bx.nb[nby];
      __builtin_amdgcn_global_load_lds((const void *)(u + oc * HALF + 4 * r), LDS_PTR(&s_o[wv][0]), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void *)(rhs + (size_t)(id - 1) * L::STRIDE + uc * HALF + 4 * r),
                                       LDS_PTR(&s_r[wv][0]), 16, 0, 0);
    }
    // (a DMA's LDS address is its wavefront's base plus the lane's slot:
    // every lane's destination below is its own slot of a 64-entry array)
    if (on && nbvx > 0) {  // the neighbour's cell across the x face
      const int p = (nbx == 0) ? NC : 1;
      __builtin_amdgcn_global_load_lds((const void *)(phi + (size_t)(nbvx - 1) * L::STRIDE + L::in_at(p, j, 0)),
                                       LDS_PTR(&s_gx[wv][0]), 4, 0, 0);
    }
    if (on && nbvx <= 0)
      __builtin_amdgcn_global_load_lds((const void *)(u + L::in_at(nbx == 0 ? 1 : NC, j, 0)), LDS_PTR(&s_x1[0][wv][0]), 4,
                                       0, 0);
    if (on && nbvy > 0 && mm == 0) {  // the neighbour's facing row of the other colour
      const int row = fy ? 1 : NC;
      __builtin_amdgcn_global_load_lds(
          (const void *)(phi + (size_t)(nbvy - 1) * L::STRIDE + oc * HALF + 4 * (row - 1)), LDS_PTR(&s_y[wv][0]), 16, 0,
          0);
    }
    if (on && nbvy <= 0)
      __builtin_amdgcn_global_load_lds((const void *)(u + L::in_at(iy, jy, 0)), LDS_PTR(&s_x1[1][wv][0]), 4, 0, 0);
    // coarse values (ghost_coarse_load's, in its order) of the items at a
    // refinement boundary
    for (int it = 0; it < 2; it++) {
      const int nb = it ? nby : nbx, nbv = it ? nbvy : nbvx, a = it ? iy : j;
      if (!(on && nbv == 0)) continue;
      const int d = nb / 2, t0 = 1 - d;
      const bool low = (nb % 2) == 0;
      const float *P = phi + (size_t)(bx.pnb[nb] - 1) * L::STRIDE;
      const int co = ((bx.ix[t0] - 1) & 1) * (NC / 2), cn = low ? NC : 1;
      auto at = [&](int qa) {
        int q[3] = {0, 0, 0};
        q[d] = cn;
        q[t0] = qa;
        return P + L::at(q[0], q[1], q[2]);
      };
      int pos[3];
      int n = 3;
      if (m.rb == RB_MG) {
        const int i = (a + 1) >> 1;
        pos[0] = co + i + 1;
        pos[1] = co + i - 1;
        pos[2] = co + i;
      } else {
        const int a1 = co + ((a + 1) >> 1);
        pos[0] = a1;
        pos[1] = a1 + 1 - 2 * (a & 1);
        pos[2] = a1;
        n = 2;
      }
      for (int v = 0; v < 3; v++)
        if (v < n) __builtin_amdgcn_global_load_lds((const void *)at(pos[v]), LDS_PTR(&s_cv[it][v][wv][0]), 4, 0, 0);
    }
    // every lane's DMAs complete before any lane reads LDS: a wavefront's
    // fence orders no DMA, and the compiler does not see the DMAs' LDS
    // writes, so the wait is explicit and keeps the reads below it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    gsync<64, 2>();
    // the ghosts of faces without a same-level neighbour (the box's second
    // cell from the face is of the other colour: in s_o)
    if (on && nbvx <= 0) {
      const float4 o = s_o[wv][lane];
      const float x2 = (nbx == 0) ? o.x : o.w;  // cell 2 or NC - 1 of the row
      CoarseVals<float> cv = {{0.0f, 0.0f, 0.0f, 0.0f, 0.0f}};
      if (nbvx == 0)
        for (int v = 0; v < 3; v++) cv.v[v] = s_cv[0][v][wv][lane];
      s_gx[wv][lane] = ghost_finish<D, NC, float>(bx, m, nbx, ghost_coarse_form<D, NC, float>(bx, m, nbx, j, 0, cv),
                                                  s_x1[0][wv][lane], x2);
    }
    if (on && nbvy <= 0) {
      const float4 o = s_o[wv][8 * bl + (fy ? NC - 2 : 1)];  // row 2 or NC - 1
      const float x2 = (mm == 0) ? o.x : (mm == 1) ? o.y : (mm == 2) ? o.z : o.w;
      CoarseVals<float> cv = {{0.0f, 0.0f, 0.0f, 0.0f, 0.0f}};
      if (nbvy == 0)
        for (int v = 0; v < 3; v++) cv.v[v] = s_cv[1][v][wv][lane];
      reinterpret_cast<float *>(&s_y[wv][8 * bl + 4 * fy])[mm] = ghost_finish<D, NC, float>(
          bx, m, nby, ghost_coarse_form<D, NC, float>(bx, m, nby, iy, 0, cv), s_x1[1][wv][lane], x2);
    }
    gsync<64, 2>();
    if (on) {
      // four cells of row j at i = i0 + 2 c; the x neighbours are the row's
      // other-colour word and its x ghost, the y neighbours the words of
      // rows j -+ 1 or the y ghosts
      const Sten<D, float> st = lpl_stencil<D, float>(bx, lambda2);
      const float4 xc = s_o[wv][lane];
      const float xe = s_gx[wv][lane];
      float xw[5];
      if (i0 == 1) {
        xw[0] = xe; xw[1] = xc.x; xw[2] = xc.y; xw[3] = xc.z; xw[4] = xc.w;
      } else {
        xw[0] = xc.x; xw[1] = xc.y; xw[2] = xc.z; xw[3] = xc.w; xw[4] = xe;
      }
      const float4 ym4 = (j == 1) ? s_y[wv][8 * bl] : s_o[wv][lane - 1];
      const float4 yp4 = (j == NC) ? s_y[wv][8 * bl + 4] : s_o[wv][lane + 1];
      const float ym[4] = {ym4.x, ym4.y, ym4.z, ym4.w}, yp[4] = {yp4.x, yp4.y, yp4.z, yp4.w};
      const float4 rv = s_r[wv][lane];
      const float rr[4] = {rv.x, rv.y, rv.z, rv.w};
      float res[4];
      if (cyl) {
        for (int c = 0; c < 4; c++) {
          float c1, c2, c3;
          cyl_coeffs<float>(bx, i0 + 2 * c, st.c, c1, c2, c3);
          const float inv1 = 1.0f / c1;
          res[c] = (rr[c] - c2 * xw[c] - c3 * xw[c + 1] - st.c[3] * ym[c] - st.c[4] * yp[c]) * inv1;
        }
      } else {
        const float inv_c1 = 1.0f / st.c[0];
        for (int c = 0; c < 4; c++)
          res[c] = (rr[c] - st.c[1] * xw[c] - st.c[2] * xw[c + 1] - st.c[3] * ym[c] - st.c[4] * yp[c]) * inv_c1;
      }
      reinterpret_cast<float4 *>(u + uc * HALF)[r] = make_float4(res[0], res[1], res[2], res[3]);
    }
    gsync<64, 2>();  // (the wavefront's LDS is reused by its next boxes)
  }
}

// k_gsrb_lds for 3D boxes of 8^3 cells in the colour-split single-precision
// layout.  A wavefront takes a box, a lane one row (j, k) of the updated
// colour (four cells, one 16-byte word): it loads its row's word of the other
// colour and of the rhs, the row's x ghost (the neighbour's cell across the
// face on the side of the row's first or last updated cell), and each of half
// the lanes one word of a y or z face (the neighbour's facing row of the other
// colour, which is the four ghosts).  On a face without a same-level
// neighbour the box's own cells next to it take the ghosts' place, and at a
// refinement boundary the coarse patches are loaded too; those ghosts are
// formed after the words are in LDS.  The y and z neighbours come from the
// other lanes' words.  The ghost and stencil expressions and their operands
// are those of k_gsrb_lds, so the results are identical.
// Four boxes per workgroup, dealt so that a workgroup's boxes come from the
// range of the list that its XCD works through (the list is ordered for one
// box per workgroup).
// Bound by its chain (record -> words -> LDS) on small levels and by the
// neighbours' scattered face words on large ones: 4096 boxes take 7.3 us
// (k_gsrb_lds: 11.9), 1024 boxes 5.2 (5.3).
template <int NC>
__global__ void __launch_bounds__(256) k_gsrb_row3d(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                    float *phi, const float *__restrict__ rhs, int redblack,
                                                    float lambda2, VarBc m, int n_boxes, int nw) {
  constexpr int D = 3;
  using L = Lay<D, NC, float>;
  using P = CoarsePatch<D, NC>;
  constexpr int HALF = L::HALF, NPT = 2 * D * P::N, NP = (NPT + 63) / 64;
  static_assert(NC == 8 && HALF == 256 && (L::STRIDE * sizeof(float)) % 16 == 0, "8^3 boxes: a row is one word");
  __shared__ float4 s_o_all[4][64];  // other colour, row (j, k) at lane (j - 1) + 8 (k - 1)
  __shared__ float4 s_f_all[4][32];  // ghosts of the faces 2 .. 5, eight rows each
  __shared__ float s_cp_all[4][NPT];
  const int wv = lgrp<64, 4>(), lane = threadIdx.x & 63;
  float4 *s_o = s_o_all[wv], *s_f = s_f_all[wv];
  float *s_cp = s_cp_all[wv];
  const int uc = redblack & 1, oc = 1 - uc;  // updated cells: (i + j + k + redblack) even
  const int j = (lane & 7) + 1, k = (lane >> 3) + 1, i0 = 1 + ((1 + j + k + uc) & 1);
  const int nbx = (i0 == 1) ? 0 : 1;  // the x face of the row's ghost
  // the y or z face row of this lane (lanes 0 .. 31): face nbf, row e
  const int nbf = 2 + ((lane >> 3) & 3), e = lane & 7, pd = (nbf & 1) ? NC : 1;
  auto row_of = [&](int p) { return nbf < 4 ? (p - 1) + NC * e : e + NC * (p - 1); };
  for (int w = blockIdx.x; w < nw; w += gridDim.x) {
    const int q = ((w >> 3) * 4 + wv) * 8 + (w & 7);
    const int id = q < n_boxes ? __builtin_amdgcn_readfirstlane(ids[q]) : 0;
    if (id <= 0) continue;  // (past the end, or a run masked out)
    const DBox &bx = boxes[id - 1];
    float *u = phi + (size_t)(id - 1) * L::STRIDE;
    int nbid[2 * D];
    bool any_rb = false, any_b = false;
#pragma unroll
    for (int nb = 0; nb < 2 * D; nb++) {
      nbid[nb] = __builtin_amdgcn_readfirstlane(bx.nb[nb]);
      any_b = any_b || nbid[nb] <= 0;
      any_rb = any_rb || nbid[nb] == 0;
    }
    const int nvx = (nbx == 0) ? nbid[0] : nbid[1], nvf = pick<2 * D>(nbid, nbf);
    const float4 xc = reinterpret_cast<const float4 *>(u + oc * HALF)[lane];
    const float4 rv = reinterpret_cast<const float4 *>(rhs + (size_t)(id - 1) * L::STRIDE + uc * HALF)[lane];
    // x ghost: the neighbour's cell, or the box's own one next to the face
    float gx = (phi + (size_t)((nvx > 0 ? nvx : id) - 1) * L::STRIDE)[L::in_at((nvx > 0) == (nbx == 0) ? NC : 1, j, k)];
    float4 fw = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (lane < 32) {
      const float *from = nvf > 0 ? phi + (size_t)(nvf - 1) * L::STRIDE + oc * HALF : u + uc * HALF;
      fw = reinterpret_cast<const float4 *>(from)[row_of((nvf > 0) == (pd == 1) ? NC : 1)];
    }
    float vp[NP];
    if (any_rb) {
      int co[3];
#pragma unroll
      for (int d = 0; d < D; d++) co[d] = ((bx.ix[d] - 1) & 1) * (NC / 2);
#pragma unroll
      for (int t = 0; t < NP; t++) {
        const int c = min(lane + t * 64, NPT - 1), nb = c / P::N, r = c % P::N, d = nb >> 1;
        const bool rb = pick<2 * D>(nbid, nb) == 0;
        int ci, cj, ck;
        face_cell<D>(nb, ((d == 0) ? co[1] : co[0]) + r % P::PP, ((d == 2) ? co[1] : co[2]) + r / P::PP,
                     (nb & 1) ? 1 : NC, ci, cj, ck);
        vp[t] = *(rb ? phi + (size_t)(pick<2 * D>(bx.pnb, nb) - 1) * L::STRIDE + L::at(ci, cj, ck) : u);
      }
    }
    const Sten<D, float> st = lpl_stencil<D, float>(bx, lambda2);
    const float inv_c1 = 1.0f / st.c[0];
    s_o[lane] = xc;
    if (any_rb)
#pragma unroll
      for (int t = 0; t < NP; t++)
        if (lane + t * 64 < NPT) s_cp[lane + t * 64] = vp[t];
    gsync<64, 4>();
    if (any_b) {
      const double run_val = m.run_val ? m.run_val[bx.run] : 0.0;
      if (nvx <= 0)
        gx = staged_ghost<D, NC, float>(bx, m, run_val, nvx, nbx, j, k, s_cp + nbx * P::N, gx, nbx == 0 ? xc.x : xc.w);
      if (lane < 32 && nvf <= 0) {
        const float4 o = s_o[row_of(pd == 1 ? 2 : NC - 1)];
        const int a0 = 1 + ((1 + pd + e + 1 + uc) & 1);
        auto ghost = [&](int c, float x1, float x2) {
          return staged_ghost<D, NC, float>(bx, m, run_val, nvf, nbf, a0 + 2 * c, e + 1, s_cp + nbf * P::N, x1, x2);
        };
        fw = make_float4(ghost(0, fw.x, o.x), ghost(1, fw.y, o.y), ghost(2, fw.z, o.z), ghost(3, fw.w, o.w));
      }
    }
    if (lane < 32) s_f[lane] = fw;
    gsync<64, 4>();
    float xw[5];
    if (i0 == 1) {
      xw[0] = gx; xw[1] = xc.x; xw[2] = xc.y; xw[3] = xc.z; xw[4] = xc.w;
    } else {
      xw[0] = xc.x; xw[1] = xc.y; xw[2] = xc.z; xw[3] = xc.w; xw[4] = gx;
    }
    const float4 ym4 = *((j == 1) ? s_f + (k - 1) : s_o + lane - 1);
    const float4 yp4 = *((j == NC) ? s_f + 8 + (k - 1) : s_o + lane + 1);
    const float4 zm4 = *((k == 1) ? s_f + 16 + (j - 1) : s_o + lane - 8);
    const float4 zp4 = *((k == NC) ? s_f + 24 + (j - 1) : s_o + lane + 8);
    const float ym[4] = {ym4.x, ym4.y, ym4.z, ym4.w}, yp[4] = {yp4.x, yp4.y, yp4.z, yp4.w};
    const float zm[4] = {zm4.x, zm4.y, zm4.z, zm4.w}, zp[4] = {zp4.x, zp4.y, zp4.z, zp4.w};
    const float rr[4] = {rv.x, rv.y, rv.z, rv.w};
    float res[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
      res[c] = (rr[c] - st.c[1] * xw[c] - st.c[2] * xw[c + 1] - st.c[3] * ym[c] - st.c[4] * yp[c] - st.c[5] * zm[c] -
                st.c[6] * zp[c]) *
               inv_c1;
    reinterpret_cast<float4 *>(u + uc * HALF)[lane] = make_float4(res[0], res[1], res[2], res[3]);
    gsync<64, 4>();  // (the wavefront's LDS is reused by its next box)
  }
}

// k_mp_residual with the box staged in LDS.
template <int D, int NC, int BS, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_mp_residual_lds(const int *__restrict__ ids,
                                                             const DBox *__restrict__ boxes,
                                                             const double *__restrict__ phi,
                                                             const double *__restrict__ rhs, float *r32, double lambda2,
                                                             int cyl, VarBc m, unsigned long long *leafmax, int nw) {
  using G = Geo<D, NC>;
  __shared__ double s_all[BB][G::NCELL];
  __shared__ double cp_all[BB][2 * D * CoarsePatch<D, NC>::N];
  double *s = s_all[lgrp<BS, BB>()], *cp = cp_all[lgrp<BS, BB>()];
  __shared__ double sh[BS / 64];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const int id = __builtin_amdgcn_readfirstlane(ids[w]);
    if (id <= 0) continue;  // run masked out
    const DBox &bx = boxes[id - 1];
    const size_t base = (size_t)(id - 1) * G::NCELL;
    constexpr int NI = (G::NINT + BS - 1) / BS;
    double rr[NI];
    for (int t = 0; t < NI; t++) {
      const int q = ltid<BS>() + t * BS;
      if (q < G::NINT) {
        int i, j, k;
        interior_ijk<D, NC>(q, i, j, k);
        rr[t] = rhs[base + G::idx(i, j, k)];
      }
    }
    Stage<D, NC, BS, double, BB, false> sg;
    sg.issue(bx, id, phi, m, 0);
    const Sten<D, double> st = lpl_stencil<D, double>(bx, lambda2);
    sg.commit(s, cp, bx, m);
    double mx = 0;
    for (int t = 0; t < NI; t++) {
      const int q = ltid<BS>() + t * BS;
      if (q >= G::NINT) break;
      int i, j, k;
      interior_ijk<D, NC>(q, i, j, k);
      const double lp = apply_cell<D, NC, double>(s, st, cyl != 0, bx, i, j, k);
      const double rv = rr[t] - lp;
      r32[(size_t)(id - 1) * Lay<D, NC, float>::STRIDE + Lay<D, NC, float>::in_at(i, j, k)] = (float)rv;
      mx = fmax(mx, fabs(rv));
    }
    if (bx.children[0] == 0) {
      mx = group_max<BS, BB>(mx, sh);
      if (ltid<BS>() == 0) atomic_max_nonneg(run_slot(leafmax, bx), mx);
    }
    gsync<BS, BB>();  // (the group's LDS is reused by its next item)
  }
}

// update_coarse, first half (m_af_multigrid.f90:703-716): per child box the
// residual rhs - L phi is restricted (with geometry) into the parent's tmp
// and phi (without geometry) into the parent's phi.  The residual is formed
// on the fly, which leaves the child's tmp untouched exactly as the
// reference's save/restore of tmp does.  With store_residual the residual is
// also kept in the child's tmp (set_coarse_phi_rhs, :742-776).
// The child box is staged in LDS with its face ghosts: formed in-kernel, or
// (stored) the stored layer, which the FP64 form fills beforehand as the
// reference does.
// OWN: every thread forms the residuals of its own cells, which then take
// phi's place in LDS for the restriction, so no thread is idle in the larger
// part: 21 M cells of 8^2 boxes 66 us (104 without), 4096 FP32 8^3 boxes 12.7
// (16.6), 64 FP64 16^3 boxes 6.2 (7.9), 768 22.0 (23.9).
// Without OWN (3D) a thread forms the residuals of the eight children of its
// parent cells and sums them in registers.  Nothing is held over a barrier,
// so a box of 16^3 needs 256 threads and a CU runs six at once, where OWN
// takes 512 threads for its residuals and runs four: FP32 levels of 512 boxes
// 7.1 us (OWN 7.9), 768 10.0 (12.1), 1536 19.2 (19.9), 2816 29.4 (32.9).
template <int D, int NC, int BS, typename T, int BB = 1, bool OWN = true>
__global__ void __launch_bounds__(BS * BB, (BS >= 512 ? 4 : 1)) k_restrict_residual(const int *__restrict__ ids,
                                                               const DBox *__restrict__ boxes, const T *child, T *phi,
                                                               const T *__restrict__ rhs, T *tmp, T lambda2, int cyl,
                                                               int store_residual, VarBc m, int stored, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  constexpr int H = NC / 2;
  constexpr int NQ = (D == 3) ? H * H * H : H * H, NQT = (NQ + BS - 1) / BS, NI = (G::NINT + BS - 1) / BS;
  static_assert(G::NINT % BS == 0, "whole strides of cells");
  __shared__ T s_all[BB][G::NCELL];
  __shared__ T cp_all[BB][2 * D * CoarsePatch<D, NC>::N];
  T *s = s_all[lgrp<BS, BB>()], *cp = cp_all[lgrp<BS, BB>()];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const int id = __builtin_amdgcn_readfirstlane(ids[w]);
    if (id <= 0) continue;  // run masked out
    const DBox &bc = boxes[id - 1];
    const DBox &bp = boxes[bc.parent - 1];
    const size_t cb = (size_t)(id - 1) * L::STRIDE, pb = (size_t)(bc.parent - 1) * L::STRIDE;
    Stage<D, NC, BS, T, BB, false> sg;
    sg.issue(bc, id, child, m, 0, (const T *)phi, stored != 0);
    T rr[OWN ? NI : 1];
    if constexpr (OWN) {
#pragma unroll
      for (int t = 0; t < NI; t++) {
        int i, j, k;
        rr[t] = rhs[cb + sg.cell(ltid<BS>() + t * BS, i, j, k)];
      }
    }
    const Sten<D, T> st = lpl_stencil<D, T>(bc, lambda2);
    sg.commit(s, cp, bc, m);
    int off[3] = {0, 0, 0};
    for (int d = 0; d < D; d++) off[d] = ((bc.ix[d] - 1) & 1) * H;
    if constexpr (OWN) {
      // the residuals of the thread's cells and its parent cells' phi
#pragma unroll
      for (int t = 0; t < NI; t++) {
        int i, j, k;
        const int pos = sg.cell(ltid<BS>() + t * BS, i, j, k);
        rr[t] = rr[t] - apply_cell<D, NC, T>(s, st, cyl != 0, bc, i, j, k);
        if (store_residual) tmp[cb + pos] = rr[t];
      }
      T ps[NQT];
#pragma unroll
      for (int t = 0; t < NQT; t++) {
        const int q = ltid<BS>() + t * BS;
        const int i = q % H + 1, j = (q / H) % H + 1, k = (D == 3) ? q / (H * H) + 1 : 0;
        if (NQ % BS == 0 || q < NQ)
          ps[t] = restrict_cell<D, NC, T>(s, 2 * i - 1, 2 * j - 1, (D == 3) ? 2 * k - 1 : 0, false, bp, 0);
      }
      gsync<BS, BB>();
#pragma unroll
      for (int t = 0; t < NI; t++) {
        int i, j, k;
        sg.cell(ltid<BS>() + t * BS, i, j, k);
        s[G::idx(i, j, k)] = rr[t];
      }
      gsync<BS, BB>();
#pragma unroll
      for (int t = 0; t < NQT; t++) {
        const int q = ltid<BS>() + t * BS;
        if (NQ % BS && q >= NQ) continue;
        const int i = q % H + 1, j = (q / H) % H + 1, k = (D == 3) ? q / (H * H) + 1 : 0;
        const int ic = off[0] + i, jc = off[1] + j, kc = (D == 3) ? off[2] + k : 0;
        tmp[pb + L::in_at(ic, jc, kc)] =
            restrict_cell<D, NC, T>(s, 2 * i - 1, 2 * j - 1, (D == 3) ? 2 * k - 1 : 0, cyl != 0, bp, ic);
        phi[pb + L::in_at(ic, jc, kc)] = ps[t];
      }
    } else {
      static_assert(D == 3, "restrict_cell's sum without cylindrical weights");
      for (int q = ltid<BS>(); q < NQ; q += BS) {
        const int i = q % H + 1, j = (q / H) % H + 1, k = q / (H * H) + 1;
        int pos[8];
        child_pos<D, NC, L>(2 * i - 1, 2 * j - 1, 2 * k - 1, pos);
        T sm = 0;  // in restrict_cell's order
#pragma unroll
        for (int c = 0; c < 8; c++) {
          const T rv = rhs[cb + pos[c]] - apply_cell<D, NC, T>(s, st, cyl != 0, bc, 2 * i - 1 + (c & 1),
                                                               2 * j - 1 + ((c >> 1) & 1), 2 * k - 1 + (c >> 2));
          if (store_residual) tmp[cb + pos[c]] = rv;
          sm = c ? sm + rv : rv;
        }
        const int to = L::in_at(off[0] + i, off[1] + j, off[2] + k);
        tmp[pb + to] = T(0.125) * sm;
        phi[pb + to] = restrict_cell<D, NC, T>(s, 2 * i - 1, 2 * j - 1, 2 * k - 1, false, bp, 0);
      }
    }
    gsync<BS, BB>();  // (the group's LDS is reused by its next item)
  }
}

// Block smoother (single-precision inner cycle only): all 2 n_cycle
// half-sweeps of one smoothing phase on a box in LDS, in one launch.  The
// values of same-level neighbour boxes are taken from `in` at the start and
// held for the whole phase (the box couples to its neighbours as in a
// block-Jacobi sweep), which lets every workgroup read `in` while writing
// `out`; physical and refinement-boundary ghosts depend on the box's own
// cells and are formed again before every half-sweep.  Inside the box the
// half-sweeps are exactly those of k_gsrb_lds.
template <int D, int NC, int BS, typename T>
__global__ void __launch_bounds__(BS) k_smooth_block(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                     const T *in, T *out, const T *__restrict__ rhs,
                                                     const T *coarse, int n_half, T lambda2, int cyl, VarBc m) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  __shared__ T s[G::NCELL];
  const int id = ids[blockIdx.x];
  if (id <= 0) return;  // run masked out
  const DBox &bx = boxes[id - 1];
  const Sten<D, T> st = lpl_stencil<D, T>(bx, lambda2);
  const size_t base = (size_t)(id - 1) * L::STRIDE;
  const T *r = rhs + base;
  lds_load_interior<D, NC, BS, T>(s, in + base);
  constexpr int NFC = 2 * D * G::NTAN;
  // same-level neighbour copies, once
  for (int q = threadIdx.x; q < NFC; q += BS) {
    const int nb = q / G::NTAN;
    if (bx.nb[nb] <= 0) continue;
    const int rr = q % G::NTAN;
    const int a = rr % NC + 1, b = (D == 3) ? rr / NC + 1 : 0;
    const bool low = (nb % 2) == 0;
    int p[3];
    face_pos<D>(nb, a, b, low ? 0 : NC + 1, p);
    s[G::idx(p[0], p[1], p[2])] = ghost_value<D, NC, T>(boxes, bx, in, m, nb, a, b, T(0), T(0));
  }
  constexpr int HALF = G::NINT / 2;
  constexpr int sx = 1, sy = G::NG, sz = G::NG * G::NG;
  for (int n = 1; n <= n_half; n++) {
    __syncthreads();
    // ghosts that depend on the box's own cells, for the colour updated now
    for (int q = threadIdx.x; q < NFC; q += BS) {
      const int nb = q / G::NTAN;
      if (bx.nb[nb] > 0) continue;
      const int rr = q % G::NTAN;
      const int a = rr % NC + 1, b = (D == 3) ? rr / NC + 1 : 0;
      const bool low = (nb % 2) == 0;
      int p[3];
      face_pos<D>(nb, a, b, low ? 1 : NC, p);
      if ((p[0] + p[1] + p[2] + n) & 1) continue;
      const T x1 = s[G::idx(p[0], p[1], p[2])];
      face_pos<D>(nb, a, b, low ? 2 : NC - 1, p);
      const T x2 = s[G::idx(p[0], p[1], p[2])];
      const T g = ghost_value<D, NC, T>(boxes, bx, in, m, nb, a, b, x1, x2, coarse);
      face_pos<D>(nb, a, b, low ? 0 : NC + 1, p);
      s[G::idx(p[0], p[1], p[2])] = g;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < HALF; q += BS) {
      const int mm = q % (NC / 2);
      const int j = (q / (NC / 2)) % NC + 1;
      const int k = (D == 3) ? q / ((NC / 2) * NC) + 1 : 0;
      const int i0 = 2 - ((n ^ (D == 3 ? k + j : j)) & 1);
      const int i = i0 + 2 * mm;
      const int x = G::idx(i, j, k);
      const T rx = r[L::in_at(i, j, k)];
      T v;
      if (D == 2) {
        if (cyl) {
          T c1, c2, c3;
          cyl_coeffs<T>(bx, i, st.c, c1, c2, c3);
          v = (rx - c2 * s[x - sx] - c3 * s[x + sx] - st.c[3] * s[x - sy] - st.c[4] * s[x + sy]) / c1;
        } else {
          v = (rx - st.c[1] * s[x - sx] - st.c[2] * s[x + sx] - st.c[3] * s[x - sy] - st.c[4] * s[x + sy]) /
              st.c[0];
        }
      } else {
        v = (rx - st.c[1] * s[x - sx] - st.c[2] * s[x + sx] - st.c[3] * s[x - sy] - st.c[4] * s[x + sy] -
             st.c[5] * s[x - sz] - st.c[6] * s[x + sz]) /
            st.c[0];
      }
      s[x] = v;
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < G::NINT; q += BS) {
    int i, j, k;
    interior_ijk<D, NC>(q, i, j, k);
    out[base + L::in_at(i, j, k)] = s[G::idx(i, j, k)];
  }
}

// phi += e on the interior of leaf boxes and e = 0 on the whole leaf box,
// ghost layer included: the refinement-boundary ghosts of finer boxes read
// a coarse leaf's ghost cells during the next cycle's first sweeps.  (Refined
// cells get the restriction of the finer phi instead, and e there is
// overwritten before the next cycle reads it.)
template <int D, int NC, int BS, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_mp_correct_leaves(const int *__restrict__ ids, double *phi, float *e,
                                                               int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, float>;
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const int id = ids[w];
    if (id <= 0) continue;  // run masked out
    double *u = phi + (size_t)(id - 1) * G::NCELL;
    float *c = e + (size_t)(id - 1) * L::STRIDE;
    // interior: the pair of cells 2s, 2s + 1 (lexicographic), one of each
    // colour, both at s in their colour's block
    for (int s = ltid<BS>(); s < L::HALF; s += BS) {
      int i, j, k;
      interior_ijk<D, NC>(2 * s, i, j, k);
      const int y = G::idx(i, j, k), c0 = (i + j + k) & 1;
      const int e0 = c0 * L::HALF + s, e1 = (1 - c0) * L::HALF + s;
      u[y] = u[y] + (double)c[e0];
      u[y + 1] = u[y + 1] + (double)c[e1];
      c[e0] = 0.0f;
      c[e1] = 0.0f;
    }
    for (int x = G::NINT + ltid<BS>(); x < G::NCELL; x += BS) c[x] = 0.0f;  // the ghosts
  }
}

// af_gc_box (afivo/src/m_af_ghostcell.f90:49-170): the face ghosts of a box
// and, with corners, its edge (3D) and corner ghosts (af_gc_box_corner
// :125-170, af_edge_gc_extrap :885-924, af_corner_gc_extrap :860-879), by one
// group of BS threads.  Only what the ghosts need is read: one value per face
// ghost (the neighbour's cell, or the box's own first one), on boxes at a
// boundary the second cells and the coarse patches too, and one value per
// edge or corner cell (the diagonal neighbour's, or the box's own cell next
// to it); all loads are in flight together.  Bound by that chain (record ->
// cells -> store), and on large levels by the scattered words of the faces
// along x.  Staging the whole box first took 9.5 us for 8 FP64 boxes of 16^3
// (now 5.2), 16.4 us for 768 (14.2), 5.2 us for 64 boxes of 8^3 (4.1), and
// 37 us a launch over the FP32 levels of 21 million 2D cells (31).
template <int D, int NC>
struct GcGeo {
  static constexpr int NTAN = Geo<D, NC>::NTAN;
  static constexpr int NFC = 2 * D * NTAN;                    // face ghosts
  static constexpr int NED = (D == 3) ? 12 * NC : 0;          // edge cells
  static constexpr int NX = NED + (1 << D);                   // and corners
};
template <int D, int NC, int BS, typename T, int BB>
__device__ inline void gc_box(T *sf, T *cp, const DBox *__restrict__ boxes, int id, T *var, const VarBc &m,
                              int corners) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  using GG = GcGeo<D, NC>;
  using P = CoarsePatch<D, NC>;
  constexpr int NTAN = G::NTAN, NF = (GG::NFC + BS - 1) / BS, NPT = 2 * D * P::N, NP = (NPT + BS - 1) / BS;
  static_assert(GG::NX <= BS, "an edge or corner cell per thread");
  const DBox &bx = boxes[id - 1];
  T *u = var + (size_t)(id - 1) * L::STRIDE;
  const int tid = ltid<BS>();
  // the thread's edge or corner cell: its direction and position
  int dir[3] = {0, 0, 0}, lo[3] = {0, 0, 0}, dim = -1, nbe = 0;
  if (corners) {
    const int e = min(tid, GG::NX - 1);
    const bool edge = e < GG::NED;
    const int n = edge ? e / NC : e - GG::NED;
    if (edge) dim = n >> 2;
    int bit = 0;
#pragma unroll
    for (int d = 0; d < D; d++) {
      const bool along = d == dim;
      const int up = (n >> bit) & 1;
      dir[d] = along ? 0 : 2 * up - 1;
      lo[d] = along ? e % NC + 1 : up ? NC + 1 : 0;
      if (!along) bit++;
    }
    nbe = bx.nbmat[nbmat_at<D>(dir[0], dir[1], dir[2])];
  }
  int nbid[2 * D];
  bool any_rb = false, any_b = false;
#pragma unroll
  for (int nb = 0; nb < 2 * D; nb++) {
    nbid[nb] = __builtin_amdgcn_readfirstlane(bx.nb[nb]);
    any_b = any_b || nbid[nb] <= 0;
    any_rb = any_rb || nbid[nb] == 0;
  }
  auto item = [&](int t, int &nb, int &a, int &b) {
    int q = tid + t * BS;
    if (GG::NFC % BS) q = min(q, GG::NFC - 1);
    nb = q / NTAN;
    a = q % NC + 1;
    b = (D == 3) ? (q % NTAN) / NC + 1 : 0;
  };
  T vf[NF], v2[NF], vp[NP];
#pragma unroll
  for (int t = 0; t < NF; t++) {
    int nb, a, b, i, j, k;
    item(t, nb, a, b);
    const int nbv = pick<2 * D>(nbid, nb);
    const bool low = (nb & 1) == 0, copy = nbv > 0;
    face_cell<D>(nb, a, b, (copy == low) ? NC : 1, i, j, k);
    vf[t] = (var + (size_t)((copy ? nbv : id) - 1) * L::STRIDE)[L::in_at(i, j, k)];
  }
  T ve = T(0);
  if (corners) {
    const int w = nbe > 0 ? NC : 1;
    ve = (var + (size_t)((nbe > 0 ? nbe : id) - 1) * L::STRIDE)[L::in_at(lo[0] - dir[0] * w, lo[1] - dir[1] * w,
                                                                         lo[2] - dir[2] * w)];
  }
  double run_val = 0.0;
  if (any_b) {
#pragma unroll
    for (int t = 0; t < NF; t++) {
      int nb, a, b, i, j, k;
      item(t, nb, a, b);
      face_cell<D>(nb, a, b, (nb & 1) ? NC - 1 : 2, i, j, k);
      v2[t] = u[L::in_at(i, j, k)];
    }
    if (any_rb) {
      int co[3];
#pragma unroll
      for (int d = 0; d < D; d++) co[d] = ((bx.ix[d] - 1) & 1) * (NC / 2);
#pragma unroll
      for (int t = 0; t < NP; t++) {
        const int q = min(tid + t * BS, NPT - 1);
        const int nb = q / P::N, e = q % P::N, d = nb >> 1;
        const bool rb = pick<2 * D>(nbid, nb) == 0;
        const int c0 = (d == 0) ? co[1] : co[0], c1 = (D == 2) ? 0 : (d == 2) ? co[1] : co[2];
        int i, j, k;
        face_cell<D>(nb, c0 + e % P::PP, (D == 3) ? c1 + e / P::PP : 0, (nb & 1) ? 1 : NC, i, j, k);
        const T *from = rb ? var + (size_t)(pick<2 * D>(bx.pnb, nb) - 1) * L::STRIDE + L::at(i, j, k) : u;
        vp[t] = *from;
      }
#pragma unroll
      for (int t = 0; t < NP; t++) {
        const int q = tid + t * BS;
        if (q < NPT) cp[q] = vp[t];
      }
      gsync<BS, BB>();
    }
    run_val = m.run_val ? m.run_val[bx.run] : 0.0;
#pragma unroll
    for (int t = 0; t < NF; t++) {
      int nb, a, b;
      item(t, nb, a, b);
      const int nbv = pick<2 * D>(nbid, nb);
      if (nbv <= 0) vf[t] = staged_ghost<D, NC, T>(bx, m, run_val, nbv, nb, a, b, cp + nb * P::N, vf[t], v2[t]);
    }
  }
#pragma unroll
  for (int t = 0; t < NF; t++) {
    const int q = tid + t * BS;
    if (GG::NFC % BS && q >= GG::NFC) continue;
    int nb, a, b, i, j, k;
    item(t, nb, a, b);
    face_cell<D>(nb, a, b, (nb & 1) ? NC + 1 : 0, i, j, k);
    u[L::at(i, j, k)] = vf[t];
    if (corners) sf[q] = vf[t];
  }
  if (!corners) {
    if (any_rb) gsync<BS, BB>();  // (cp is reused by the group's next item)
    return;
  }
  gsync<BS, BB>();
  if (tid < GG::NX) {
    // the face ghost next to the cell along axis d: at p, behind the face of
    // axis f
    auto ghost = [&](int f, int p0, int p1, int p2) {
      const int df = (f == 0) ? dir[0] : (f == 1) ? dir[1] : dir[2];
      const int a = (f == 0) ? p1 : p0, b = (D == 2) ? 1 : (f == 2) ? p1 : p2;
      return sf[(2 * f + (df > 0)) * NTAN + (a - 1) + NC * (b - 1)];
    };
    const int x = lo[0], y = lo[1], z = lo[2], xi = x - dir[0], yi = y - dir[1], zi = z - dir[2];
    if (nbe <= 0) {
      if (D == 2) {
        ve = ghost(1, xi, y, 0) + ghost(0, x, yi, 0) - ve;
      } else if (dim >= 0) {
        // moved inwards along axis dim + 1 (behind the face of axis
        // dim + 2), then along axis dim + 2
        const int o0 = (dim == 2) ? 0 : dim + 1, o1 = (dim == 0) ? 2 : dim - 1;
        const T g0 = ghost(o1, o0 == 0 ? xi : x, o0 == 1 ? yi : y, o0 == 2 ? zi : z);
        const T g1 = ghost(o0, o1 == 0 ? xi : x, o1 == 1 ? yi : y, o1 == 2 ? zi : z);
        ve = g0 + g1 - ve;
      } else {
        ve = ghost(0, x, yi, zi) + ghost(1, xi, y, zi) + ghost(2, xi, yi, z) - 2 * ve;
      }
    }
    u[L::at(x, y, z)] = ve;
  }
  gsync<BS, BB>();  // (the group's LDS is reused by its next item)
}
template <int D, int NC, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_gc(const int *__restrict__ ids, const DBox *__restrict__ boxes, T *var,
                                                    VarBc m, int corners, int nw) {
  __shared__ T s_all[BB][GcGeo<D, NC>::NFC];
  __shared__ T cp_all[BB][2 * D * CoarsePatch<D, NC>::N];
  T *s = s_all[lgrp<BS, BB>()], *cp = cp_all[lgrp<BS, BB>()];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const int id = __builtin_amdgcn_readfirstlane(ids[w]);
    if (id <= 0) continue;  // run masked out
    gc_box<D, NC, BS, T, BB>(s, cp, boxes, id, var, m, corners);
  }
}

// k_gc with corners on a level, and k_coarse_rhs on its boxes with children:
// the two that follow the restriction onto a level, in one launch (the
// second reads only its own box's cells and the ghosts just filled).  Both
// are bound by their chains on small levels of 2D boxes.
template <int D, int NC, int BS, typename T, int BB = 1>
__global__ void __launch_bounds__(BS * BB) k_gc_rhs(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                    T *phi, T *rhs, T *tmp, T lambda2, int cyl, int copy_phi,
                                                    VarBc m, int nw) {
  using G = Geo<D, NC>;
  using L = Lay<D, NC, T>;
  __shared__ T s_all[BB][GcGeo<D, NC>::NFC];
  __shared__ T cp_all[BB][2 * D * CoarsePatch<D, NC>::N];
  T *s = s_all[lgrp<BS, BB>()], *cp = cp_all[lgrp<BS, BB>()];
  for (int w = item0<BS, BB>(); w < nw; w += item_stride<BB>()) {
    const int id = __builtin_amdgcn_readfirstlane(ids[w]);
    if (id <= 0) continue;  // run masked out
    const DBox &bx = boxes[id - 1];
    const size_t base = (size_t)(id - 1) * L::STRIDE;
    const bool parent = bx.children[0] > 0;
    gc_box<D, NC, BS, T, BB>(s, cp, boxes, id, phi, m, 1);
    if (!parent) continue;
    // (the ghosts were stored by other threads of the group)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    gsync<BS, BB>();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    const Sten<D, T> st = lpl_stencil<D, T>(bx, lambda2);
#pragma unroll 2
    for (int x = ltid<BS>(); x < G::NCELL; x += BS) {
      int i, j, k;
      bool inner;
      if constexpr (L::SPLIT) {
        inner = x < G::NINT;
        if (inner) colour_cell<D, NC>(x >= L::HALF, x >= L::HALF ? x - L::HALF : x, i, j, k);
      } else {
        i = x % G::NG, j = (x / G::NG) % G::NG, k = (D == 3) ? x / (G::NG * G::NG) : 0;
        inner = i >= 1 && i <= NC && j >= 1 && j <= NC && (D == 2 || (k >= 1 && k <= NC));
      }
      // (nothing reads the ghost part of a split pool's rhs)
      if (inner)
        rhs[base + x] = apply_cell<D, NC, T, L>(phi + base, st, cyl != 0, bx, i, j, k) + tmp[base + x];
      else if (!L::SPLIT)
        rhs[base + x] = rhs[base + x] + tmp[base + x];
      if (copy_phi) tmp[base + x] = phi[base + x];
    }
  }
}

// The same for several FP64 variables in one launch: work item w is box
// w / vars.n, variable w % vars.n.
constexpr int GC_MAX_VARS = 8;
struct GcVars {
  double *v[GC_MAX_VARS];
  VarBc m[GC_MAX_VARS];
  int n;
};
template <int D, int NC, int BS>
__global__ void __launch_bounds__(BS) k_gc_vars(const int *__restrict__ ids, const DBox *__restrict__ boxes,
                                                    GcVars vars, int corners, int nw) {
  __shared__ double s[GcGeo<D, NC>::NFC];
  __shared__ double cp[2 * D * CoarsePatch<D, NC>::N];
  for (int w = blockIdx.x; w < nw; w += gridDim.x) {
    const int id = ids[w / vars.n];
    if (id <= 0) continue;
    gc_box<D, NC, BS, double, 1>(s, cp, boxes, id, vars.v[w % vars.n], vars.m[w % vars.n], corners);
  }
}

}  // namespace afg
