// The segmented y-line Chebyshev step: residual and both Thomas sweeps of every
// line in one pass, each line split into segments of a few rows, one per thread.
// Shared by the single-case kernels (pp_mg.hip) and the batched ones (pp_batch.hip).
#pragma once

#include "pp_mg_dev.hpp"

namespace pp {

// FP32 levels keep, besides the planar FP16 coefficients, the three 8-byte records the
// step reads per cell (launch_line_pack): pi = [g11 g12 g13 | class byte],
// pk = [g31 g32 g33 g21], pj = [g22 g23 | inv].  A row then takes five wide loads (its
// own three records, pi of the west neighbour, pk of the k - 1 neighbour) where the
// planar arrays take seventeen narrow ones, and the loaded values wait for their use
// packed, in 10 registers instead of 17.
template <typename T>
struct LineRowIn;

template <>
struct LineRowIn<float> {
  u32x2 i0, j0, k0;  // own records
  u32x2 iw, km;      // pi of the west cell, pk of the k - 1 cell
  float f;
  float xp[5], xc[4];
};
template <>
struct LineRowIn<double> {
  double g[9], gw[3], gb[3];
  double inv, f;
  uint8_t cl;
  double xp[5], xc[4];
};

__device__ __forceinline__ _Float16 lo_half(uint32_t v) {
  const uint16_t b = (uint16_t)(v & 0xffffu);
  return __builtin_bit_cast(_Float16, b);
}
__device__ __forceinline__ _Float16 hi_half(uint32_t v) {
  const uint16_t b = (uint16_t)(v >> 16);
  return __builtin_bit_cast(_Float16, b);
}

// element type of a level's coefficients
template <typename T>
struct LineCoef {
  using type = double;
};
template <>
struct LineCoef<float> {
  using type = _Float16;
};

__device__ __forceinline__ void line_coef(const LineRowIn<float>& r, const _Float16 (&gs_prev)[3],
                                          RowCoef<_Float16>& rc, float& inv, bool& interior) {
  rc.v[0][0] = lo_half(r.i0.x); rc.v[0][1] = hi_half(r.i0.x); rc.v[0][2] = lo_half(r.i0.y);
  rc.v[1][0] = lo_half(r.iw.x); rc.v[1][1] = hi_half(r.iw.x); rc.v[1][2] = lo_half(r.iw.y);
  rc.v[2][0] = hi_half(r.k0.y); rc.v[2][1] = lo_half(r.j0.x); rc.v[2][2] = hi_half(r.j0.x);
  rc.v[4][0] = lo_half(r.k0.x); rc.v[4][1] = hi_half(r.k0.x); rc.v[4][2] = lo_half(r.k0.y);
  rc.v[5][0] = lo_half(r.km.x); rc.v[5][1] = hi_half(r.km.x); rc.v[5][2] = lo_half(r.km.y);
#pragma unroll
  for (int e = 0; e < 3; e++) rc.v[3][e] = gs_prev[e];
  inv = __uint_as_float(r.j0.y);
  interior = ((r.i0.y >> 16) & CLS_INTERIOR) != 0;
}
__device__ __forceinline__ void line_coef(const LineRowIn<double>& r, const double (&gs_prev)[3],
                                          RowCoef<double>& rc, double& inv, bool& interior) {
#pragma unroll
  for (int e = 0; e < 3; e++) {
    rc.v[0][e] = r.g[e];
    rc.v[1][e] = r.gw[e];
    rc.v[2][e] = r.g[3 + e];
    rc.v[3][e] = gs_prev[e];
    rc.v[4][e] = r.g[6 + e];
    rc.v[5][e] = r.gb[e];
  }
  inv = r.inv;
  interior = (r.cl & CLS_INTERIOR) != 0;
}

// upper j-face coefficients of cell c
__device__ __forceinline__ void line_gs(const LevelView<float>& L, uint32_t c, _Float16 (&g)[3]) {
  const u32x2 k = ld_at(L.pk, c), j = ld_at(L.pj, c);
  g[0] = hi_half(k.y);
  g[1] = lo_half(j.x);
  g[2] = hi_half(j.x);
}
__device__ __forceinline__ void line_gs(const LevelView<double>& L, uint32_t c, double (&g)[3]) {
  const size_t n = L.d.n();
#pragma unroll
  for (int e = 0; e < 3; e++) g[e] = ld_at(L.g + (size_t)(3 + e) * n, c);
}

// The row's SP and NP coefficients (build_row's accumulation order) from its faces:
// the tridiagonal part of A along j.  The step forms a_j and cp_j = c_j inv_j from
// them instead of reading the Thomas factors' a and cp.
template <typename T, typename TG>
__device__ __forceinline__ void line_ac_interior(const RowCoef<TG>& rc, T& a, T& c) {
  const T q = T(0.25);
  const T e = q * (T)rc.v[1][1] - q * (T)rc.v[0][1];
  const T kc = q * (T)rc.v[4][1], kb = q * (T)rc.v[5][1];
  a = ((e + (T)rc.v[3][1]) - kc) + kb;
  c = (((T)rc.v[2][1] - e) + kc) - kb;
}
template <int D, int SGN, typename T, typename TG>
__device__ __forceinline__ void line_ac_cross(const RowCoef<TG>& rc, uint32_t code, T& a, T& c) {
  // a face across i or k: its j-difference reaches SP and NP
  constexpr int F = 2 * D + (SGN > 0 ? 0 : 1);
  constexpr int XI = D == 0 ? 0 : 1;
  const int cc = (int)((code >> (6 + 4 * F + 2 * XI)) & 3u);
  const bool on = ((code >> F) & 1u) != 0;
  const T g = on ? (T)rc.v[F][1] : T(0);
  const T whi = cc == X_CENTRAL ? T(0.25) : (cc == X_UPPER ? T(0.5) : T(0));
  const T wlo = cc == X_CENTRAL ? T(0.25) : (cc == X_LOWER ? T(0.5) : T(0));
  a += (SGN > 0 ? -wlo : wlo) * g;
  c += (SGN > 0 ? whi : -whi) * g;
}
template <int SGN, typename T, typename TG>
__device__ __forceinline__ T line_ac_j(const RowCoef<TG>& rc, uint32_t code) {
  // a j face: its normal term, and the (c, q) part of its one-sided cross terms
  constexpr int F = SGN > 0 ? 2 : 3;
  if (!((code >> F) & 1u)) return T(0);
  T v = (T)rc.v[F][1];
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const int cc = (int)((code >> (6 + 4 * F + 2 * e)) & 3u);
    const T wmd = cc == X_LOWER ? T(0.5) : (cc == X_UPPER ? T(-0.5) : T(0));
    v += (SGN > 0 ? wmd : -wmd) * (T)rc.v[F][e == 0 ? 0 : 2];
  }
  return v;
}
template <typename T, typename TG>
__device__ __forceinline__ void line_ac_coded(const RowCoef<TG>& rc, uint32_t code, T& a, T& c) {
  a = c = T(0);
  line_ac_cross<0, +1>(rc, code, a, c);
  line_ac_cross<0, -1>(rc, code, a, c);
  a += line_ac_j<-1, T>(rc, code);
  c += line_ac_j<+1, T>(rc, code);
  line_ac_cross<2, +1>(rc, code, a, c);
  line_ac_cross<2, -1>(rc, code, a, c);
  if (!(code & ROW_BIT)) a = c = T(0);
}

// a[off bytes] from a base all lanes share
template <typename T>
__device__ __forceinline__ T ld_b(const T* __restrict__ a, uint32_t off) {
  typedef const __attribute__((address_space(1))) char gchar;
  typedef const __attribute__((address_space(1))) T gT;
  return *(gT*)((gchar*)a + off);
}

// LDS of one block: per sweep, every segment's zero-carry end value and multiplier
// product (two sweeps, so a block going round for its next tile needs no extra barrier)
template <typename T, int S, int LANES>
struct LineLds {
  T part[2][2][S][LANES];
};

// One layout of the step: W waves and LANES lines per block, S = W * 64 / LANES segments
// per line of up to LM rows.  KEEP: what the walk over the rows leaves in registers.
//   0 the residual (a and 1 / den are read after the walk, cp and x with them);
//   1 the upward sweep's two values per row (cp and x are read after the walk);
//   2 those, cp and x (nothing is read twice).
// LM and KEEP are bounded by registers.  In FP32 every layout stays within the 128 that
// leave four waves per SIMD (88 to 114 for a step from x, 94 to 120 batched).  In FP64
// they do not all: 146, 131, 158 and 200 registers in layouts 0, 1, 3 and 5 (3, 3, 3 and 2
// waves per SIMD), and the 1024-thread blocks of layouts 2 and 4 are held to 128 and spill
// 4 and 2 (batched 8 and 12); they are still the faster ones where line_layout picks them.
template <int LM_, int W_, int LANES_, int KEEP_>
struct LineLayout {
  static constexpr int LM = LM_, W = W_, LANES = LANES_, S = W_ * 64 / LANES_, KEEP = KEEP_;
};
// Calls fn with layout y's LineLayout (see line_layout, and batch_line_layout for BATCHED)
template <typename T, bool BATCHED = false, typename F>
inline void with_line_layout(int y, F&& fn) {
  if constexpr (std::is_same<T, float>::value) {
    switch (y) {
      case 0: fn(LineLayout<4, 4, 16, 2>{}); break;
      case 1: fn(LineLayout<4, 8, 32, 2>{}); break;
      case 2: fn(LineLayout<8, 8, 32, 2>{}); break;
      case 3: fn(LineLayout<8, 16, 64, 2>{}); break;
      case 4: fn(LineLayout<8, 8, 16, 2>{}); break;
      case 5: fn(LineLayout<16, 8, 32, 1>{}); break;
      default: fn(LineLayout<16, 16, 64, 1>{});
    }
  } else {
    if constexpr (BATCHED) {
      if (y == 6) return fn(LineLayout<8, 4, 16, 0>{});
      if (y == 7) return fn(LineLayout<16, 4, 16, 0>{});
    }
    switch (y) {
      case 0: fn(LineLayout<4, 4, 16, 2>{}); break;
      case 1: fn(LineLayout<8, 8, 16, 0>{}); break;
      case 2: fn(LineLayout<8, 16, 64, 0>{}); break;
      case 3: fn(LineLayout<12, 4, 16, 0>{}); break;
      case 4: fn(LineLayout<8, 16, 32, 0>{}); break;
      default: fn(LineLayout<16, 8, 32, 0>{});
    }
  }
}

// fn(0), fn(1), ... for the first min(nr, N) row numbers, as constants
template <int Q, int N, typename F>
__device__ __forceinline__ void for_rows(int nr, F&& fn) {
  if constexpr (Q < N) {
    if (Q < nr) {
      fn(std::integral_constant<int, Q>{});
      for_rows<Q + 1, N>(nr, fn);
    }
  }
}

// One Chebyshev step in three-term form on the lines this block holds:
// z = T^-1 (f - A x), x_new = x + c1 (x - x_prev) + c2 z (x_prev null: zero; x_new may
// be x_prev's buffer).  Each thread walks the rows of its segment upwards.  It keeps x
// in the five columns (i, k), (i +- 1, k), (i, k +- 1) for the rows below, at and above
// the current one, so a row loads five values of x for the row above and the four
// (i +- 1, k +- 1) ones of its own row (9 instead of 19), and the row's lower j-face
// coefficients are the row below's upper ones.
//
// The sweeps are affine recurrences, d_j = (r_j - a_j d_{j-1}) inv_j upwards and
// z_j = d_j - cp_j z_{j+1} downwards.  The upward one runs along with the walk from a
// zero carry, keeping d_j and the product P_j of the multipliers; the carry C into the
// segment is then added as d_j + P_j C.  The downward one does the same.  The
// coefficients are used where they are loaded, a_j and cp_j come from the row's own
// faces, and nothing is computed twice.  Carries: every wave chains the end values of
// the segments before its own from LDS (one barrier per sweep).
//
// Every thread of the block must call it; lanes without a line pass live = false and
// read line (i, k) = (0, 0).
template <typename T, typename Y, int MODE>
__device__ __forceinline__ void line_step(const LevelView<T>& L, bool live, int i, int k, const T* __restrict__ f,
                                          const T* __restrict__ lfac, const T* __restrict__ x_old, const T* x_prev,
                                          T* x_new, T c1, T c2, LineLds<T, Y::S, Y::LANES>& sh) {
  using TG = typename LineCoef<T>::type;
  constexpr int LM = Y::LM, LANES = Y::LANES, S = Y::S;
  constexpr int KEEP = MODE == LS_ZERO ? 0 : Y::KEEP;
  constexpr uint32_t B = sizeof(T);
  const Dims& d = L.d;
  const size_t n = d.n();
  const int lane = (int)(threadIdx.x & (LANES - 1));
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  const int rows = (d.ny + S - 1) / S;
  // first row of this wave's (first) segment, and its row count
  const int jw = wv * (64 / LANES) * rows;
  const int nrw = max(0, min(rows, d.ny - jw));
  const int s = LANES == 64 ? wv : wv * (64 / LANES) + (int)threadIdx.x / LANES;
  const int nr = LANES == 64 ? nrw : max(0, min(rows, d.ny - s * rows));
  const uint32_t nx = (uint32_t)d.nx, plane = nx * (uint32_t)d.ny;
  // a lane in the wave's second segment starts `rows` rows above the first; its rows
  // past the last one are read at the last one (jrel: the lane's row offset)
  const int jrel = LANES == 64 ? 0 : s * rows - jw;
  const int jlast = d.ny - 1;
  const uint32_t ic = (uint32_t)i, kc = (uint32_t)k * plane;
  const uint32_t base = ic + kc;
  const T* __restrict__ linv = lfac + 2 * n;
  // row q of the segment, split into a part all lanes share (an element offset) and
  // the lane's own (0 for 64-lane layouts)
  auto row_of = [&](int q, uint32_t& su, uint32_t& sl) {
    if constexpr (LANES == 64) {
      su = (uint32_t)min(jw + q, jlast) * nx;
      sl = 0;
    } else {
      su = 0;
      sl = (uint32_t)min(jw + jrel + q, jlast) * nx;
    }
  };

  T dl[LM], P[LM], cp[LM], xs[LM];
#pragma unroll
  for (int q = 0; q < LM; q++) dl[q] = P[q] = cp[q] = xs[q] = T(0);
  T dend = T(0), prod = T(1);
  auto up = [&](int q, T r, T a, T inv) {
    const T v = (r - a * dend) * inv, p = prod * -(a * inv);
    if (LANES == 64 || q < nr) {
      dend = v;
      prod = p;
    }
    dl[q] = dend;
    P[q] = prod;
  };
  if constexpr (MODE == LS_ZERO) {
#pragma unroll
    for (int q = 0; q < LM; q++)
      if (q < nrw) {
        uint32_t su, sl;
        row_of(q, su, sl);
        dl[q] = ld_b(f + su, (base + sl) * B);
      }
  } else if (nrw > 0) {
    const uint32_t ip = (uint32_t)wrap_p(i, d.nx, d.per[0]), im = (uint32_t)wrap_m(i, d.nx, d.per[0]);
    const uint32_t kp = (uint32_t)wrap_p(k, d.nz, d.per[2]) * plane, km = (uint32_t)wrap_m(k, d.nz, d.per[2]) * plane;
    // columns C, E, W, T, B (marched) and TE, BE, TW, BW (read at the row itself)
    const uint32_t col[5] = {base, ip + kc, im + kc, ic + kp, ic + km};
    const uint32_t cor[4] = {ip + kp, ip + km, im + kp, im + km};
    auto load_row = [&](int q, LineRowIn<T>& r) {
      uint32_t su, sl, pu, pl;
      row_of(q, su, sl);
      row_of(q + 1, pu, pl);
      if constexpr (std::is_same<T, float>::value) {
        r.i0 = ld_b(L.pi + su, (col[0] + sl) * 8u);
        r.k0 = ld_b(L.pk + su, (col[0] + sl) * 8u);
        r.j0 = ld_b(L.pj + su, (col[0] + sl) * 8u);
        r.iw = ld_b(L.pi + su, (col[2] + sl) * 8u);
        r.km = ld_b(L.pk + su, (col[4] + sl) * 8u);
      } else {
#pragma unroll
        for (int e = 0; e < 9; e++) r.g[e] = ld_b(L.g + (size_t)e * n + su, (col[0] + sl) * 8u);
#pragma unroll
        for (int e = 0; e < 3; e++) {
          r.gw[e] = ld_b(L.g + (size_t)e * n + su, (col[2] + sl) * 8u);
          r.gb[e] = ld_b(L.g + (size_t)(6 + e) * n + su, (col[4] + sl) * 8u);
        }
        r.inv = KEEP == 0 ? 0. : ld_b(linv + su, (col[0] + sl) * 8u);
        r.cl = ld_b(L.cls + su, col[0] + sl);
      }
      r.f = MODE == LS_POWER ? T(0) : ld_b(f + su, (col[0] + sl) * B);
#pragma unroll
      for (int e = 0; e < 5; e++) r.xp[e] = ld_b(x_old + pu, (col[e] + pl) * B);
#pragma unroll
      for (int e = 0; e < 4; e++) r.xc[e] = ld_b(x_old + su, (cor[e] + sl) * B);
    };
    T xm[5], x0[5];
    TG gs_prev[3];
    {
      uint32_t su, sl;
      row_of(0, su, sl);
      const uint32_t mu = LANES == 64 ? (uint32_t)max(jw - 1, 0) * nx : 0u;
      const uint32_t ml = LANES == 64 ? 0u : (uint32_t)max(min(jw + jrel, jlast) - 1, 0) * nx;
#pragma unroll
      for (int e = 0; e < 5; e++) {
        xm[e] = ld_b(x_old + mu, (col[e] + ml) * B);
        x0[e] = ld_b(x_old + su, (col[e] + sl) * B);
      }
      line_gs(L, base + mu + ml, gs_prev);
    }
    LineRowIn<T> r;
    load_row(0, r);
    for_rows<0, LM>(nrw, [&](auto qc) __attribute__((always_inline)) {
      constexpr int q = decltype(qc)::value;
      T xv[19];
      xv[CP] = x0[0]; xv[NP] = r.xp[0]; xv[SP] = xm[0];
      xv[EP] = x0[1]; xv[NE] = r.xp[1]; xv[SE] = xm[1];
      xv[WP] = x0[2]; xv[NW] = r.xp[2]; xv[SW] = xm[2];
      xv[TP] = x0[3]; xv[TN] = r.xp[3]; xv[TS] = xm[3];
      xv[BP] = x0[4]; xv[BN] = r.xp[4]; xv[BS] = xm[4];
      xv[TE] = r.xc[0];
      xv[BE] = r.xc[1];
      xv[TW] = r.xc[2];
      xv[BW] = r.xc[3];
      RowCoef<TG> rc;
      T inv, ax, dg, a, c;
      bool interior, row = true;
      line_coef(r, gs_prev, rc, inv, interior);
      if (__all(interior)) {
        flux_row_v<X_CENTRAL>(rc, CODE_INTERIOR, xv, ax, dg);
        line_ac_interior(rc, a, c);
      } else {
        uint32_t su, sl;
        row_of(q, su, sl);
        const uint32_t cd = ld_b(L.code + su, (base + sl) * 4u);
        flux_row_v<-1>(rc, cd, xv, ax, dg);
        line_ac_coded(rc, cd, a, c);
        row = (cd & ROW_BIT) != 0;
      }
      if constexpr (std::is_same<T, float>::value) {
        ax *= L.gs;
        a *= L.gs;
        c *= L.gs;
      }
      if constexpr (KEEP == 0) dl[q] = row ? r.f - ax : T(0);
      else up(q, row ? r.f - ax : T(0), a, inv);
      if constexpr (KEEP == 2) {
        cp[q] = c * inv;
        xs[q] = x0[0];
      }
#pragma unroll
      for (int e = 0; e < 5; e++) {
        xm[e] = x0[e];
        x0[e] = r.xp[e];
      }
#pragma unroll
      for (int e = 0; e < 3; e++) gs_prev[e] = rc.v[2][e];
      if constexpr (q + 1 < LM) load_row(q + 1, r);
    });
  }
  if constexpr (KEEP == 0) {
    T aa[LM], vv[LM];
#pragma unroll
    for (int q = 0; q < LM; q++) {
      aa[q] = vv[q] = T(0);
      if (q < nrw) {
        uint32_t su, sl;
        row_of(q, su, sl);
        const uint32_t o = (base + sl) * B;
        aa[q] = ld_b(lfac + su, o);
        vv[q] = ld_b(linv + su, o);
      }
    }
#pragma unroll
    for (int q = 0; q < LM; q++)
      if (q < nrw) up(q, dl[q], aa[q], vv[q]);
  }
  sh.part[0][0][s][lane] = dend;
  sh.part[0][1][s][lane] = prod;
  // the downward sweep's operands, in flight across the barrier
  const bool rd = MODE == LS_NEXT && c1 != T(0) && x_prev;
  T xq[LM];
#pragma unroll
  for (int q = 0; q < LM; q++) {
    xq[q] = T(0);
    if (q < nrw) {
      uint32_t su, sl;
      row_of(q, su, sl);
      const uint32_t o = (base + sl) * B;
      if constexpr (KEEP != 2) {
        cp[q] = ld_b(lfac + n + su, o);
        if constexpr (MODE == LS_NEXT) xs[q] = ld_b(x_old + su, o);
      }
      if (rd) xq[q] = ld_b(x_prev + su, o);
    }
  }
  __syncthreads();
  T carry = T(0);
#pragma unroll 4
  for (int t = 0; t < s; t++) carry = sh.part[0][0][t][lane] + sh.part[0][1][t][lane] * carry;
  T zend = T(0);
  prod = T(1);
#pragma unroll
  for (int q = LM - 1; q >= 0; q--)
    if (q < nrw) {
      const T v = (dl[q] + P[q] * carry) - cp[q] * zend, p = prod * -cp[q];
      if (LANES == 64 || q < nr) {
        zend = v;
        prod = p;
      }
      dl[q] = zend;
      P[q] = prod;
    }
  sh.part[1][0][s][lane] = zend;
  sh.part[1][1][s][lane] = prod;
  __syncthreads();
  carry = T(0);
#pragma unroll 4
  for (int t = S - 1; t > s; t--) carry = sh.part[1][0][t][lane] + sh.part[1][1][t][lane] * carry;
#pragma unroll
  for (int q = 0; q < LM; q++)
    if (q < nr && live) {
      uint32_t su, sl;
      row_of(q, su, sl);
      const T z = dl[q] + P[q] * carry;
      T* o = reinterpret_cast<T*>(reinterpret_cast<char*>(x_new + su) + (base + sl) * B);
      if constexpr (MODE == LS_POWER) *o = z;
      else if constexpr (MODE == LS_ZERO) *o = c2 * z;
      else *o = xs[q] + (c1 * (xs[q] - xq[q]) + c2 * z);
    }
}

}  // namespace pp
