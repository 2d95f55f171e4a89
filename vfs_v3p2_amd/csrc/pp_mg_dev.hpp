// Device bodies of the multigrid kernels: Chebyshev smoothers, fused residual +
// restriction, IB-masked prolongation and the dense coarsest solve.  Each body
// takes explicit cell (or tile) coordinates, so the single-case kernels
// (pp_mg.hip) and the batched persistent kernels (pp_batch.hip) share the
// arithmetic.
//
// The transfers follow the reference's MG primitives (MyRestriction
// poisson.c:364-471, MyInterpolation poisson.c:473-669): restriction sums the
// fluid children of a coarse cell (the coarse operator is in the same integrated
// flux form as the fine one, so coarse residuals add up), zero on coarse IB
// cells; prolongation uses the (27,9,9,3,9,3,3,1)/64 weights, one-sided next to
// coarse IB cells and at non-periodic walls, periodic axes wrap.
#pragma once

#include <type_traits>

#include "pp_kernels.hpp"
#include "pp_pair_dev.hpp"
#include "pp_stencil.hpp"

namespace pp {

// (A x)_c and the diagonal on a level, from its coefficients in either storage
template <typename T>
__device__ __forceinline__ void level_flux(const LevelView<T>& L, uint32_t cd, size_t c, const Nbr& nb,
                                           const T (&xv)[19], T& ax, T& diag) {
  if constexpr (std::is_same<T, float>::value) {
    if (L.gh) {
      flux_row(L.gh, L.d.n(), cd, c, nb.s[WP], nb.s[SP], nb.s[BP], xv, ax, diag);
      ax *= L.gs;
      diag *= L.gs;
      return;
    }
  }
  flux_row(L.g, L.d.n(), cd, c, nb.s[WP], nb.s[SP], nb.s[BP], xv, ax, diag);
}

// D^-1 of the level operator, 0 on cells that carry no unknown.
template <typename T>
__device__ __forceinline__ void dinv_cell(const LevelView<T>& L, T* __restrict__ dinv, int i, int j, int k) {
  const size_t c = L.d.idx(i, j, k);
  const uint32_t cd = L.code[c];
  Nbr nb;
  neighbours(L.d, i, j, k, nb);
  T xv[19];
#pragma unroll
  for (int s = 0; s < 19; s++) xv[s] = T(0);
  T ax, diag;
  level_flux(L, cd, c, nb, xv, ax, diag);
  dinv[c] = ((cd & ROW_BIT) && diag != T(0)) ? T(1) / diag : T(0);
}

// (A x)_c, the diagonal and whether the cell has a row, with the level's class
// bytes picking the row form: a wave whose cells are all interior (class flag)
// takes the compile-time-weight form and reads no code word.  The coefficient
// loads are issued before the class test, together with the caller's stencil
// loads.
template <typename T, typename TG>
__device__ __forceinline__ void flux_by_class(const TG* __restrict__ g, size_t n, const uint32_t* __restrict__ code,
                                              size_t c, const Nbr& nb, const T (&xv)[19], bool interior, T& ax,
                                              T& diag, bool& row) {
  RowCoef<TG> rc;
  load_coef(g, n, (uint32_t)c, nb.s[WP], nb.s[SP], nb.s[BP], rc);
  if (__all(interior)) {
    flux_row_v<X_CENTRAL>(rc, CODE_INTERIOR, xv, ax, diag);
  } else {
    const uint32_t cd = code[c];
    flux_row_v<-1>(rc, cd, xv, ax, diag);
    row = (cd & ROW_BIT) != 0;
  }
}

// Chebyshev smoothing preconditioned by the diagonal, in three-term form: one step is
//   z = D^-1 (f - A x);  x_new = x + c1 (x - x_prev) + c2 z
// (the direction d = x - x_prev is not stored; c1 == 0 starts a new sequence and
// does not read x_prev).  x_new may be x_prev's buffer.  Modes:
//   SM_NEXT    one step from x_old;
//   SM_ZERO    the first step from x = 0:  x_new = c2 D^-1 f, x_prev = 0;
//   SM_FIRST2  the first two steps from x = 0 in one pass: the first step's
//              x1 = c0 D^-1 f is formed on the fly at the 19 neighbours from f and
//              D^-1 (or from fd = f D^-1 when the writer of f stored it), then one
//              step from x1 with (c1, c2); x_new = x2, x_prev = x1;
//   SM_POWER   dv = D^-1 (f - A x_old) only.
// The level's class bytes pick the row form: a wave whose cells are all interior
// takes the compile-time-weight form and reads no code word.  g holds the
// level's coefficients in their storage type (FP16 scaled by gs, or T); every
// load of the cell -- class, f, x_prev, the 19 stencil values, the 18
// coefficients -- is issued before any of them is used.
template <typename T, int MODE, typename TG>
__device__ __forceinline__ void smooth_point_body(const LevelView<T>& L, const TG* __restrict__ g, bool scaled,
                                                  const T* __restrict__ f, const T* __restrict__ dinv,
                                                  const T* __restrict__ x_old, T* x_prev, T* x_new,
                                                  T* __restrict__ dv, T c1, T c2, T c0, int i, int j, int k,
                                                  const T* __restrict__ fd) {
  const size_t c = L.d.idx(i, j, k);
  const uint8_t cl = L.cls[c];
  const T fc = f[c];
  T xp = T(0);
  if constexpr (MODE == SM_NEXT) {
    if (c1 != T(0)) xp = x_prev[c];
  }
  Nbr nb;
  neighbours(L.d, i, j, k, nb);
  T xv[19];
  if constexpr (MODE == SM_FIRST2) {
    if (fd) {
#pragma unroll
      for (int s = 0; s < 19; s++) xv[s] = c0 * fd[nb.s[s]];
    } else {
#pragma unroll
      for (int s = 0; s < 19; s++) xv[s] = c0 * (f[nb.s[s]] * dinv[nb.s[s]]);
    }
  } else {
    load_x(nb, x_old, xv);
  }
  T ax, diag;
  bool row = true;
  flux_by_class(g, L.d.n(), L.code, c, nb, xv, (cl & CLS_INTERIOR) != 0, ax, diag, row);
  if (scaled) {
    ax *= L.gs;
    diag *= L.gs;
  }
  // straight-line division with a safe divisor: a branch around it would let the
  // compiler move the load of f into the branch, after the stencil
  const bool live = row && diag != T(0);
  const T z = live ? (fc - ax) / (live ? diag : T(1)) : T(0);
  if constexpr (MODE == SM_POWER) {
    dv[c] = z;
    return;
  }
  const T xc = xv[CP];
  const T dold = (MODE == SM_FIRST2) ? xc : (c1 == T(0) ? T(0) : xc - xp);
  if constexpr (MODE == SM_FIRST2) x_prev[c] = row ? xc : T(0);
  x_new[c] = row ? xc + (c1 * dold + c2 * z) : T(0);
}

template <typename T, int MODE>
__device__ __forceinline__ void smooth_point_cell(const LevelView<T>& L, const T* __restrict__ f,
                                                  const T* __restrict__ dinv, const T* __restrict__ x_old,
                                                  T* x_prev, T* x_new, T* __restrict__ dv, T c1, T c2, T c0, int i,
                                                  int j, int k, const T* __restrict__ fd = nullptr) {
  if constexpr (MODE == SM_ZERO) {
    const size_t c = L.d.idx(i, j, k);
    x_new[c] = c2 * (f[c] * dinv[c]);
    x_prev[c] = T(0);
    return;
  } else {
    if constexpr (std::is_same<T, float>::value) {
      if (L.gh) {
        smooth_point_body<T, MODE>(L, L.gh, true, f, dinv, x_old, x_prev, x_new, dv, c1, c2, c0, i, j, k, fd);
        return;
      }
    }
    smooth_point_body<T, MODE>(L, L.g, false, f, dinv, x_old, x_prev, x_new, dv, c1, c2, c0, i, j, k, fd);
  }
}

// (A x) and the diagonal on a pair from x already loaded, with the class bytes picking the
// row form (see flux_by_class); row: which of the two cells have one
template <typename T, typename TG>
__device__ __forceinline__ void pair_by_class(const LevelView<T>& L, const TG* __restrict__ g, bool scaled,
                                              const PairAt& at, PairX<T>& xs, T (&ax)[2], T (&dg)[2],
                                              bool (&row)[2]) {
  uint8_t cl[2];
  PairG<TG> gs;
  ld_pair(L.cls, at.c, cl);
  pair_load_g(at, g, L.d.n(), gs);
  pair_share_x(at, xs);
  pair_share_g(at, gs);
  row[0] = row[1] = true;
  if (__all((cl[0] & CLS_INTERIOR) && (cl[1] & CLS_INTERIOR))) {
    const uint32_t cd[2] = {CODE_INTERIOR, CODE_INTERIOR};
    pair_flux<X_CENTRAL>(gs, xs, cd, ax, dg);
  } else {
    uint32_t cd[2];
    ld_pair(L.code, at.c, cd);
    pair_flux<-1>(gs, xs, cd, ax, dg);
    row[0] = (cd[0] & ROW_BIT) != 0;
    row[1] = (cd[1] & ROW_BIT) != 0;
  }
  if (scaled) {
#pragma unroll
    for (int m = 0; m < 2; m++) ax[m] *= L.gs, dg[m] *= L.gs;
  }
}

// smooth_point_cell on a pair of cells of an FP64 level (SM_NEXT, SM_FIRST2)
template <typename T, int MODE>
__device__ __forceinline__ void smooth_point_pair(const LevelView<T>& L, const T* __restrict__ f,
                                                  const T* __restrict__ dinv, const T* __restrict__ x_old,
                                                  T* x_prev, T* x_new, T c1, T c2, T c0, const PairAt& at,
                                                  const T* __restrict__ fd) {
  static_assert(std::is_same<T, double>::value, "FP32 levels take one cell per thread (launch_smooth)");
  T fc[2], xp[2] = {T(0), T(0)}, xn[2];
  PairX<T> xs;
  ld_pair(f, at.c, fc);
  if constexpr (MODE == SM_NEXT) {
    if (c1 != T(0)) ld_pair((const T*)x_prev, at.c, xp);
    pair_load_x(at, x_old, xs);
  } else {
    pair_load_x(at, fd ? fd : f, xs);
    if (fd) {
#pragma unroll
      for (int s = 0; s < 9; s++) xs.v[s][0] *= c0, xs.v[s][1] *= c0;
#pragma unroll
      for (int s = 0; s < 5; s++) xs.l[s] *= c0, xs.r[s] *= c0;
    } else {
      PairX<T> ds;
      pair_load_x(at, dinv, ds);
#pragma unroll
      for (int s = 0; s < 9; s++)
        xs.v[s][0] = c0 * (xs.v[s][0] * ds.v[s][0]), xs.v[s][1] = c0 * (xs.v[s][1] * ds.v[s][1]);
#pragma unroll
      for (int s = 0; s < 5; s++) xs.l[s] = c0 * (xs.l[s] * ds.l[s]), xs.r[s] = c0 * (xs.r[s] * ds.r[s]);
    }
  }
  T ax[2], dg[2];
  bool row[2];
  pair_by_class(L, L.g, false, at, xs, ax, dg, row);
#pragma unroll
  for (int m = 0; m < 2; m++) {
    const bool live = row[m] && dg[m] != T(0);
    const T z = live ? (fc[m] - ax[m]) / (live ? dg[m] : T(1)) : T(0);
    const T xc = xs.v[0][m];
    const T dold = MODE == SM_FIRST2 ? xc : (c1 == T(0) ? T(0) : xc - xp[m]);
    xn[m] = row[m] ? xc + (c1 * dold + c2 * z) : T(0);
  }
  if constexpr (MODE == SM_FIRST2)
    st_pair(x_prev, at.c, at.both, row[0] ? xs.v[0][0] : T(0), row[1] ? xs.v[0][1] : T(0));
  st_pair(x_new, at.c, at.both, xn[0], xn[1]);
}

// Thomas factors of the y-line tridiagonal part of A on the line (i, k), from the
// rows' SP / CP / NP coefficients (cells without an unknown get the identity):
// lfac = [a | cp | inv], each n long; den_j = b_j - a_j cp_{j-1}, inv_j = 1/den_j,
// cp_j = c_j inv_j.  First pass, one thread per cell: the row's (a, b, c) into
// lfac's three parts.
template <typename T>
__device__ __forceinline__ void line_rows_cell(const LevelView<T>& L, T* __restrict__ lfac, int i, int j, int k) {
  const size_t n = L.d.n();
  const size_t c = L.d.idx(i, j, k);
  const uint32_t cd = L.code[c];
  T a = T(0), b = T(1), cc = T(0);
  if (cd & ROW_BIT) {
    Nbr nb;
    neighbours(L.d, i, j, k, nb);
    T vol[19];
    if (L.gh) {
      build_row(L.gh, n, cd, c, nb.s[WP], nb.s[SP], nb.s[BP], vol);
      a = vol[SP] * L.gs;
      b = vol[CP] * L.gs;
      cc = vol[NP] * L.gs;
    } else {
      build_row(L.g, n, cd, c, nb.s[WP], nb.s[SP], nb.s[BP], vol);
      a = vol[SP];
      b = vol[CP];
      cc = vol[NP];
    }
  }
  lfac[c] = a;
  lfac[n + c] = b;
  lfac[2 * n + c] = cc;
}

// The factorisation along the line (i, k), in place over line_rows_cell's rows:
// den_j = b_j - a_j cp_{j-1}, inv_j = 1 / den_j (0 when den_j is 0), cp_j = c_j inv_j.
// The rows' loads do not depend on the recurrence, so eight rows are loaded at a time.
template <typename T>
__device__ __forceinline__ void line_factors_col(const Dims& d, T* __restrict__ lfac, int i, int k) {
  const size_t n = d.n();
  const size_t sy = (size_t)d.nx;
  const size_t c0 = d.idx(i, 0, k);
  T cprev = T(0);
  constexpr int LC = 8;
  for (int j0 = 0; j0 < d.ny; j0 += LC) {
    T b[LC], cc[LC], a[LC];
#pragma unroll
    for (int q = 0; q < LC; q++) {
      a[q] = b[q] = cc[q] = T(0);
      if (j0 + q < d.ny) {
        const size_t c = c0 + (size_t)(j0 + q) * sy;
        a[q] = lfac[c];
        b[q] = lfac[n + c];
        cc[q] = lfac[2 * n + c];
      }
    }
#pragma unroll
    for (int q = 0; q < LC; q++) {
      if (j0 + q < d.ny) {
        const size_t c = c0 + (size_t)(j0 + q) * sy;
        const T den = b[q] - a[q] * cprev;
        const T inv = den != T(0) ? T(1) / den : T(0);
        cprev = cc[q] * inv;
        lfac[n + c] = cprev;
        lfac[2 * n + c] = inv;
      }
    }
  }
}

// r = f - A x on cells with an unknown, 0 elsewhere.  The class byte picks the
// row form (interior waves read no code word); every load is issued before the
// vote.
template <typename T, typename TG>
__device__ __forceinline__ void resid_body(const LevelView<T>& L, const TG* __restrict__ g, bool scaled,
                                           const T* __restrict__ f, const T* __restrict__ x, T* __restrict__ r,
                                           int i, int j, int k) {
  const size_t c = L.d.idx(i, j, k);
  const uint8_t cl = L.cls[c];
  const T fc = f[c];
  Nbr nb;
  neighbours(L.d, i, j, k, nb);
  T xv[19], ax, dg;
  load_x(nb, x, xv);
  bool row = true;
  flux_by_class(g, L.d.n(), L.code, c, nb, xv, (cl & CLS_INTERIOR) != 0, ax, dg, row);
  if (scaled) ax *= L.gs;
  r[c] = row ? fc - ax : T(0);
}

template <typename T>
__device__ __forceinline__ void resid_cell(const LevelView<T>& L, const T* __restrict__ f, const T* __restrict__ x,
                                           T* __restrict__ r, int i, int j, int k) {
  if constexpr (std::is_same<T, float>::value) {
    if (L.gh) {
      resid_body(L, L.gh, true, f, x, r, i, j, k);
      return;
    }
  }
  resid_body(L, L.g, false, f, x, r, i, j, k);
}

// what a y-line step computes: LS_ZERO the step from x = 0 (r = f); LS_NEXT a step from
// x_old; LS_POWER z alone, to x_new (the power iteration)
enum { LS_NEXT = 0, LS_ZERO = 1, LS_POWER = 2 };

// One Chebyshev step preconditioned by the y-line tridiagonal part T of A on the
// line (i, k), in three-term form: z = T^-1 r with the precomputed factors (forward
// sweep parked in tmp), x_new = x + c1 (x - x_prev) + c2 z (x_prev null: zero; x_new may
// be x_prev's buffer).  For lines too long for the segmented step (pp_line_dev.hpp).
// The line is walked in chunks of LC rows whose inputs are loaded into registers
// first (independent loads in flight together), then the recurrence runs on them:
// the sequential sweep is otherwise bound by one load latency per row.
template <typename T, int MODE>
__device__ __forceinline__ void line_solve_col(const Dims& d, const T* __restrict__ r, const T* __restrict__ lfac,
                                               T* __restrict__ tmp, const T* __restrict__ x_old, const T* x_prev,
                                               T* x_new, T c1, T c2, int i, int k) {
  constexpr int LC = 16;
  const size_t n = d.n();
  const T* __restrict__ la = lfac;
  const T* __restrict__ lcp = lfac + n;
  const T* __restrict__ linv = lfac + 2 * n;
  const size_t sy = (size_t)d.nx;
  const size_t c0 = d.idx(i, 0, k);
  const int ny = d.ny;
  T dprev = T(0);
  for (int j0 = 0; j0 < ny; j0 += LC) {
    T rr[LC], aa[LC], vv[LC];
#pragma unroll
    for (int q = 0; q < LC; q++) {
      const int j = j0 + q < ny ? j0 + q : ny - 1;  // clamped rows are loaded but not used
      const size_t c = c0 + (size_t)j * sy;
      rr[q] = r[c];
      aa[q] = la[c];
      vv[q] = linv[c];
    }
#pragma unroll
    for (int q = 0; q < LC; q++) {
      if (j0 + q < ny) {
        dprev = (rr[q] - aa[q] * dprev) * vv[q];
        tmp[c0 + (size_t)(j0 + q) * sy] = dprev;
      }
    }
  }
  T znext = T(0);
  const bool rd = MODE == LS_NEXT && c1 != T(0) && x_prev;
  for (int j1 = ny - 1; j1 >= 0; j1 -= LC) {
    T tt[LC], pp[LC], xq[LC], xo[LC];
#pragma unroll
    for (int q = 0; q < LC; q++) {
      const int j = j1 - q >= 0 ? j1 - q : 0;
      const size_t c = c0 + (size_t)j * sy;
      tt[q] = tmp[c];
      pp[q] = lcp[c];
      xq[q] = rd ? x_prev[c] : T(0);
      xo[q] = MODE == LS_NEXT ? x_old[c] : T(0);
    }
#pragma unroll
    for (int q = 0; q < LC; q++) {
      if (j1 - q >= 0) {
        const size_t c = c0 + (size_t)(j1 - q) * sy;
        const T z = tt[q] - pp[q] * znext;
        znext = z;
        x_new[c] = MODE == LS_POWER ? z : (MODE == LS_ZERO ? c2 * z : xo[q] + (c1 * (xo[q] - xq[q]) + c2 * z));
      }
    }
  }
}

// fc[C] = sum over fluid children of (f - A x); zero on coarse IB cells.  Any
// coarsening mask; one thread per coarse cell.
template <typename T>
__device__ __forceinline__ void resid_restrict_cell(const LevelView<T>& F, const T* __restrict__ f,
                                                    const T* __restrict__ x, const Dims& dc,
                                                    const uint8_t* __restrict__ clsc, int cmask, T* __restrict__ fc,
                                                    int ic, int jc, int kc) {
  const size_t C = dc.idx(ic, jc, kc);
  if (clsc[C] & CLS_NONFLUID) { fc[C] = T(0); return; }
  const int i0 = (cmask & 1) ? 2 * ic : ic, i1 = (cmask & 1) ? min(2 * ic + 1, F.d.nx - 1) : ic;
  const int j0 = (cmask & 2) ? 2 * jc : jc, j1 = (cmask & 2) ? min(2 * jc + 1, F.d.ny - 1) : jc;
  const int k0 = (cmask & 4) ? 2 * kc : kc, k1 = (cmask & 4) ? min(2 * kc + 1, F.d.nz - 1) : kc;
  T sum = T(0);
  for (int k = k0; k <= k1; k++)
    for (int j = j0; j <= j1; j++)
      for (int i = i0; i <= i1; i++) {
        const size_t c = F.d.idx(i, j, k);
        const uint32_t cd = F.code[c];
        if (!(cd & ROW_BIT)) continue;
        Nbr nb;
        neighbours(F.d, i, j, k, nb);
        T xv[19], ax, dg;
        load_x(nb, x, xv);
        level_flux(F, cd, c, nb, xv, ax, dg);
        sum += f[c] - ax;
      }
  fc[C] = sum;
}

// fc[C] from the fine residual r (f - A x on the rows, as resid_cell writes it): the
// sum resid_restrict_cell forms, over the same children in the same (k, j, i) order,
// rows only, zero on coarse IB cells -- the same value to the last bit, with the
// children's residuals computed one thread per fine cell beforehand.
template <typename T>
__device__ __forceinline__ void restrict_sum_cell(const LevelView<T>& F, const T* __restrict__ r, const Dims& dc,
                                                  const uint8_t* __restrict__ clsc, int cmask, T* __restrict__ fc,
                                                  int ic, int jc, int kc) {
  const size_t C = dc.idx(ic, jc, kc);
  if (clsc[C] & CLS_NONFLUID) { fc[C] = T(0); return; }
  const int i0 = (cmask & 1) ? 2 * ic : ic, i1 = (cmask & 1) ? min(2 * ic + 1, F.d.nx - 1) : ic;
  const int j0 = (cmask & 2) ? 2 * jc : jc, j1 = (cmask & 2) ? min(2 * jc + 1, F.d.ny - 1) : jc;
  const int k0 = (cmask & 4) ? 2 * kc : kc, k1 = (cmask & 4) ? min(2 * kc + 1, F.d.nz - 1) : kc;
  T sum = T(0);
  for (int k = k0; k <= k1; k++)
    for (int j = j0; j <= j1; j++)
      for (int i = i0; i <= i1; i++) {
        const size_t c = F.d.idx(i, j, k);
        if (F.code[c] & ROW_BIT) sum += r[c];
      }
  fc[C] = sum;
}

// Residual + restriction when all three axes are coarsened, for the 64x2x2 fine
// tile (bx, by, bz) of a (64,2,2) block: one thread per fine cell, pair sums in i
// by lane shuffle, the j and k pairs through LDS; the tile covers coarse cells
// (32 bx .. 32 bx + 31, by, bz).  Every thread of the block must call it.
template <typename T>
__device__ __forceinline__ void resid_restrict_blk(const LevelView<T>& F, const T* __restrict__ f,
                                                   const T* __restrict__ x, const Dims& dc,
                                                   const uint8_t* __restrict__ clsc, T* __restrict__ fc, int bx,
                                                   int by, int bz, bool keep_y, T (*lds)[2][32]) {
  const int tx = threadIdx.x, ty = threadIdx.y, tz = threadIdx.z;
  const int i = bx * 64 + tx, j = by * 2 + ty, k = bz * 2 + tz;
  T r = T(0);
  if (i < F.d.nx && j < F.d.ny && k < F.d.nz) {
    const size_t c = F.d.idx(i, j, k);
    const uint32_t cd = F.code[c];
    Nbr nb;
    neighbours(F.d, i, j, k, nb);
    T xv[19], ax, dg;
    load_x(nb, x, xv);
    level_flux(F, cd, c, nb, xv, ax, dg);
    if (cd & ROW_BIT) r = f[c] - ax;
  }
  r += __shfl_xor(r, 1, 64);
  if ((tx & 1) == 0) lds[tz][ty][tx >> 1] = r;
  __syncthreads();
  if (keep_y) {
    // i and k coarsened only: the two j rows of the tile are two coarse cells
    if (tz == 0 && tx < 32) {
      const int ic = bx * 32 + tx, jc = by * 2 + ty, kc = bz;
      if (ic < dc.nx && jc < dc.ny && kc < dc.nz) {
        const size_t C = dc.idx(ic, jc, kc);
        const T v = lds[0][ty][tx] + lds[1][ty][tx];
        fc[C] = (clsc[C] & CLS_NONFLUID) ? T(0) : v;
      }
    }
  } else if (ty == 0 && tz == 0 && tx < 32) {
    const int ic = bx * 32 + tx, jc = by, kc = bz;
    if (ic < dc.nx && jc < dc.ny && kc < dc.nz) {
      const size_t C = dc.idx(ic, jc, kc);
      const T v = (lds[0][0][tx] + lds[0][1][tx]) + (lds[1][0][tx] + lds[1][1][tx]);
      fc[C] = (clsc[C] & CLS_NONFLUID) ? T(0) : v;
    }
  }
  __syncthreads();  // the LDS tile is reused by the block's next tile
}

// f - A x on a pair's rows, 0 elsewhere and on a first cell that is another thread's
template <typename T>
__device__ __forceinline__ T resid_pair_sum(const LevelView<T>& L, const T* __restrict__ f, const T* __restrict__ x,
                                            const PairAt& at) {
  T fc[2], ax[2], dg[2];
  bool row[2];
  PairX<T> xs;
  ld_pair(f, at.c, fc);
  pair_load_x(at, x, xs);
  if constexpr (std::is_same<T, float>::value) {
    if (L.gh) pair_by_class(L, L.gh, true, at, xs, ax, dg, row);
    else pair_by_class(L, L.g, false, at, xs, ax, dg, row);
  } else {
    pair_by_class(L, L.g, false, at, xs, ax, dg, row);
  }
  const T r0 = (at.both && row[0]) ? fc[0] - ax[0] : T(0), r1 = row[1] ? fc[1] - ax[1] : T(0);
  return r0 + r1;
}

// Coarse cells of one block of resid_restrict_pairs
HDI uint32_t restrict_tile(bool keep_y) { return keep_y ? 128u : 64u; }

// Residual + restriction as in resid_restrict_blk (the same sums in the same order) for
// tile `tile` of the level's coarse cells in flat order, so levels of any width fill every
// lane: a thread takes the two children adjacent in i, the block's four waves the two or
// four rows of them (j kept: two rows, 128 coarse cells).  Every thread of the 256-thread
// block must call it.
template <typename T>
__device__ __forceinline__ void resid_restrict_pairs(const LevelView<T>& F, const T* __restrict__ f,
                                                     const T* __restrict__ x, const Dims& dc,
                                                     const uint8_t* __restrict__ clsc, T* __restrict__ fc,
                                                     uint32_t tile, bool keep_y, T (*lds)[2][64]) {
  const int lane = threadIdx.x & 63, lo = (threadIdx.x >> 6) & 1, hi = threadIdx.x >> 7;
  const uint32_t E = keep_y ? tile * 128u + 64u * lo + lane : tile * 64u + lane;
  int ic, jc, kc;
  const bool in = flat_cell(dc, E, ic, jc, kc);
  T r = T(0);
  if (in) {
    const int j = keep_y ? jc : 2 * jc + lo, k = 2 * kc + hi;
    if (j < F.d.ny && k < F.d.nz) r = resid_pair_sum(F, f, x, pair_at(F.d, ic, j, k));
  }
  lds[hi][lo][lane] = r;
  __syncthreads();
  if (in && hi == 0 && (keep_y || lo == 0)) {
    const T v = keep_y ? lds[0][lo][lane] + lds[1][lo][lane]
                       : (lds[0][0][lane] + lds[0][1][lane]) + (lds[1][0][lane] + lds[1][1][lane]);
    fc[E] = (clsc[E] & CLS_NONFLUID) ? T(0) : v;
  }
  __syncthreads();  // the LDS tile is reused by the block's next tile
}

__device__ __forceinline__ int axis_pick(int f, int n, int per, bool coarsened, int& ic) {
  if (!coarsened) { ic = f; return 0; }
  ic = f >> 1;
  int ia = (f & 1) ? 1 : -1;
  if (!per && (f == 0 || f == n - 1)) ia = 0;
  return ia;
}
__device__ __forceinline__ int wrapc(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// xf += P xc at fine cell (i, j, k): trilinear (27,9,9,3,9,3,3,1)/64, one-sided
// next to coarse IB cells (poisson.c:500-505; the three neighbour tests are
// independent).  Every operand is loaded at once - the fine mask, the three
// coarse neighbours' masks and the coarse values at both choices on each axis
// (cached) - and the one-sided choice is a register select, so the cell costs
// one round trip to memory instead of three.
template <typename T>
__device__ __forceinline__ void prolong_add_cell(const LevelView<T>& F, const Dims& dc,
                                                 const uint8_t* __restrict__ clsc, int cmask,
                                                 const T* __restrict__ xc, T* __restrict__ xf, int i, int j, int k) {
  const size_t c = F.d.idx(i, j, k);
  int ic, jc, kc;
  const int ia = axis_pick(i, F.d.nx, F.d.per[0], cmask & 1, ic);
  const int ja = axis_pick(j, F.d.ny, F.d.per[1], cmask & 2, jc);
  const int ka = axis_pick(k, F.d.nz, F.d.per[2], cmask & 4, kc);
  const int in = wrapc(ic + ia, dc.nx), jn = wrapc(jc + ja, dc.ny), kn = wrapc(kc + ka, dc.nz);
  const uint8_t fm = F.cls[c];
  const uint8_t mk = clsc[dc.idx(ic, jc, kn)], mj = clsc[dc.idx(ic, jn, kc)], mi = clsc[dc.idx(in, jc, kc)];
  const T x000 = xc[dc.idx(ic, jc, kc)], x010 = xc[dc.idx(ic, jn, kc)];
  const T x100 = xc[dc.idx(in, jc, kc)], x110 = xc[dc.idx(in, jn, kc)];
  const T x001 = xc[dc.idx(ic, jc, kn)], x011 = xc[dc.idx(ic, jn, kn)];
  const T x101 = xc[dc.idx(in, jc, kn)], x111 = xc[dc.idx(in, jn, kn)];
  const T xo = xf[c];
  // neighbour used on each axis: the other coarse cell unless the axis is not
  // coarsened, the cell sits on a non-periodic wall, or that coarse cell is IB
  const bool ui = ia != 0 && !(mi & CLS_NONFLUID);
  const bool uj = ja != 0 && !(mj & CLS_NONFLUID);
  const bool uk = ka != 0 && !(mk & CLS_NONFLUID);
  const T y0 = uj ? x010 : x000, y1 = uj ? x110 : x100;  // (ic, j2, kc), (in, j2, kc)
  const T z0 = uj ? x011 : x001, z1 = uj ? x111 : x101;  // (ic, j2, kn), (in, j2, kn)
  const T a_c = x000, a_j = y0, a_i = ui ? x100 : x000, a_ij = ui ? y1 : y0;
  const T b_c = uk ? x001 : a_c, b_j = uk ? z0 : a_j;
  const T b_i = uk ? (ui ? x101 : x001) : a_i, b_ij = uk ? (ui ? z1 : z0) : a_ij;
  const T v = (a_c * T(9) + a_j * T(3) + a_i * T(3) + a_ij) * T(3. / 64.) +
              (b_c * T(9) + b_j * T(3) + b_i * T(3) + b_ij) * T(1. / 64.);
  if (!(fm & CLS_NONFLUID)) xf[c] = xo + v;
}

// What the prolongation walks: coarse columns by fine rows where i is coarsened, else the
// fine cells
HDI Dims prolong_dims(const Dims& fine, const Dims& coarse, int cmask) {
  Dims d = fine;
  if (cmask & 1) d.nx = coarse.nx;
  return d;
}

// prolong_add_cell (the same terms in the same order) on the one or two fine cells of
// coarse column ic in fine row (j, k), axis i coarsened.  The two share the parent, the j
// and k picks and their masks, and the parent's four coarse values, so a pair decides and
// computes little more than a cell did: the cell form kept the vector units 75% busy at a
// quarter of HBM's rate (FP32 levels of 512x256x256 167 -> 114 us, 256x128x128 42 -> 29,
// 192x96x128 14.4 -> 9.6).
template <typename T>
__device__ __forceinline__ void prolong_add_pair(const LevelView<T>& F, const Dims& dc,
                                                 const uint8_t* __restrict__ clsc, int cmask,
                                                 const T* __restrict__ xc, T* __restrict__ xf, int ic, int j, int k) {
  const int i = 2 * ic;
  const uint32_t c = (uint32_t)F.d.idx(i, j, k);
  const bool two = i + 1 < F.d.nx;
  int jc, kc;
  const int ja = axis_pick(j, F.d.ny, F.d.per[1], cmask & 2, jc);
  const int ka = axis_pick(k, F.d.nz, F.d.per[2], cmask & 4, kc);
  const int jn = wrapc(jc + ja, dc.ny), kn = wrapc(kc + ka, dc.nz);
  const uint32_t im = (uint32_t)wrapc(ic - 1, dc.nx), ip = (uint32_t)wrapc(ic + 1, dc.nx), in = (uint32_t)ic;
  const uint32_t r00 = (uint32_t)dc.idx(0, jc, kc), r10 = (uint32_t)dc.idx(0, jn, kc),
                 r01 = (uint32_t)dc.idx(0, jc, kn), r11 = (uint32_t)dc.idx(0, jn, kn);
  const uint8_t mk = ld_at(clsc, r01 + in), mj = ld_at(clsc, r10 + in), ml = ld_at(clsc, r00 + im),
                mr = ld_at(clsc, r00 + ip);
  T p[4], l[4], r[4], xo[2] = {T(0), T(0)};
  uint8_t fm[2] = {0, CLS_NONFLUID};
  const uint32_t row[4] = {r00, r10, r01, r11};
#pragma unroll
  for (int q = 0; q < 4; q++) {
    p[q] = ld_at(xc, row[q] + in);
    l[q] = ld_at(xc, row[q] + im);
    r[q] = ld_at(xc, row[q] + ip);
  }
  fm[0] = ld_at(F.cls, c);
  xo[0] = ld_at((const T*)xf, c);
  if (two) {
    fm[1] = ld_at(F.cls, c + 1);
    xo[1] = ld_at((const T*)xf, c + 1);
  }
  const bool uj = ja != 0 && !(mj & CLS_NONFLUID);
  const bool uk = ka != 0 && !(mk & CLS_NONFLUID);
  const T a_c = p[0], a_j = uj ? p[1] : p[0];
  const T b_c = uk ? p[2] : a_c, b_j = uk ? (uj ? p[3] : p[2]) : a_j;
#pragma unroll
  for (int m = 0; m < 2; m++) {
    const T(&n)[4] = m ? r : l;
    const bool wall = !F.d.per[0] && (m ? i + 1 == F.d.nx - 1 : (i == 0 || i == F.d.nx - 1));
    const bool ui = !wall && !((m ? mr : ml) & CLS_NONFLUID);
    const T a_i = ui ? n[0] : a_c, a_ij = ui ? (uj ? n[1] : n[0]) : a_j;
    const T b_i = uk ? (ui ? n[2] : p[2]) : a_i, b_ij = uk ? (ui ? (uj ? n[3] : n[2]) : b_j) : a_ij;
    const T v = (a_c * T(9) + a_j * T(3) + a_i * T(3) + a_ij) * T(3. / 64.) +
                (b_c * T(9) + b_j * T(3) + b_i * T(3) + b_ij) * T(1. / 64.);
    if (!(fm[m] & CLS_NONFLUID)) xf[c + m] = xo[m] + v;
  }
}

// x = Cinv f for rows DENSE_ROWS rb .. DENSE_ROWS rb + DENSE_ROWS - 1, Cinv column-major
// n x n (n <= 1024): the 256 threads of a block are 32 rows x 8 column chains (chain ch
// takes columns ch, ch + 8, ...), whose sums meet in LDS.  Every thread must call it.
// Bound by memory latency: a thread's loads are issued 16 columns ahead of their use,
// the first ones before f is staged, and 32-row blocks spread a 512-row matrix over 16
// CUs (512 rows: 31 -> 9 us in FP32, 23.8 -> 8.8 us in FP64 against 64-row blocks with
// two loads in flight).
constexpr int DENSE_ROWS = 32;
template <typename T>
__device__ __forceinline__ void dense_rows(int n, const T* __restrict__ cinv, const T* __restrict__ f,
                                           T* __restrict__ x, int rb, T* fs, T (*part)[DENSE_ROWS]) {
  constexpr int U = 16;
  const int row = threadIdx.x & (DENSE_ROWS - 1), ch = threadIdx.x / DENSE_ROWS;
  const int r = rb * DENSE_ROWS + row;
  const T* __restrict__ col = cinv + (r < n ? r : 0);
  T v[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int c = ch + 8 * u;
    v[u] = c < n ? col[(size_t)c * n] : T(0);
  }
  for (int t = threadIdx.x; t < n && t < 1024; t += 256) fs[t] = f[t];
  __syncthreads();
  T a = T(0);
  for (int c0 = ch; c0 < n; c0 += 8 * U) {
    T w[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int c = c0 + 8 * (U + u);
      w[u] = c < n ? col[(size_t)c * n] : T(0);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int c = c0 + 8 * u;
      if (c < n) a += v[u] * fs[c];
    }
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = w[u];
  }
  part[ch][row] = a;
  __syncthreads();
  // chains ch and ch + 4 are one quarter of the columns (the coarse tail's order)
  if (ch == 0 && r < n)
    x[r] = ((part[0][row] + part[4][row]) + (part[1][row] + part[5][row])) +
           ((part[2][row] + part[6][row]) + (part[3][row] + part[7][row]));
  __syncthreads();  // fs and part are reused by the block's next tile
}

}  // namespace pp
