// The 19-point operator on two cells adjacent in i per thread, from 16-byte (FP64) or
// 8-byte (FP32) loads.
//
// A CU's L1 serves a wave's load at 16 lanes per clock when a lane asks for 4 bytes and at
// 4 lanes per clock when it asks for 8 or 16 (measured: 4.6, 16.1 and 16.2 clocks per wave
// load), so one cell per thread bounds an FP64 stencil by its 39 8-byte loads a row, far
// under HBM's rate.  Two cells share one 16-byte load of every coefficient and stencil row,
// the index arithmetic, the face between them, and ten of their stencil values.  What lies
// beyond the pair, x at i - 1 and i + 2 and the i - 1/2 face's coefficients, comes from the
// neighbouring lanes; a lane whose neighbour does not hold it loads it.
//
// A row of odd length ends in a pair that overlaps the one before: both compute that cell,
// one stores it.
#pragma once

#include "pp_common.hpp"
#include "pp_stencil.hpp"

namespace pp {

// two entries at an index of either parity (rows of odd length start at one)
template <typename T>
struct Pair2;
template <>
struct Pair2<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };
template <>
struct Pair2<float> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <>
struct Pair2<_Float16> { typedef _Float16 type __attribute__((ext_vector_type(2), aligned(2))); };
template <>
struct Pair2<uint32_t> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(4))); };
template <>
struct Pair2<uint8_t> { typedef uint8_t type __attribute__((ext_vector_type(2), aligned(1))); };

template <typename T>
__device__ __forceinline__ void ld_pair(const T* __restrict__ a, uint32_t idx, T (&v)[2]) {
  typedef typename Pair2<T>::type P;
  typedef const __attribute__((address_space(1))) char gchar;
  typedef const __attribute__((address_space(1))) P gP;
  const P p = *(gP*)((gchar*)a + idx * (uint32_t)sizeof(T));
  v[0] = p.x;
  v[1] = p.y;
}
// both entries, or only the second where the first is another thread's
template <typename T>
__device__ __forceinline__ void st_pair(T* __restrict__ a, uint32_t idx, bool both, T v0, T v1) {
  typedef typename Pair2<T>::type P;
  if (both) *(P*)(a + idx) = P{v0, v1};
  else a[idx + 1] = v1;
}

// Pairs of a row (levels of at least two cells in i)
HDI int pairs_of(int nx) { return (nx + 1) >> 1; }
HDI uint32_t pair_count(const Dims& d) { return (uint32_t)pairs_of(d.nx) * (uint32_t)d.ny * (uint32_t)d.nz; }
HDI Dims pair_dims(const Dims& d) {
  Dims p = d;
  p.nx = pairs_of(d.nx);
  return p;
}

// Fewer cells than this take one cell per thread in a single case's kernels: the chip is not
// full and a call lasts as long as one thread's arithmetic (24^3: 3.5 against 4.2 us for A x,
// 64^3: 6.8 against 5.6).  The batched operator and restriction always take pairs, so that a
// member's sums do not depend on the members beside it (a batch of one 24^3: the same 1.03-
// 1.10 ms either way, its restriction being one launch instead of two).
constexpr uint32_t PAIR_MIN_CELLS = 1u << 16;
HDI bool takes_pairs(size_t cells) { return cells >= PAIR_MIN_CELLS; }

// Rows per slab of the pair walk.  A k plane of the FP64 operator's operands is re-read for
// the next plane's k-1/2 faces and stencil; planes of more than about 16k cells outgrow an
// XCD's L2, so they are walked in slabs of about that many (512x256x256, A x: 672 us in
// whole planes, 674 / 642 / 659 in slabs of 8k / 16k / 32k cells).
HDI uint32_t pair_slab(const Dims& d) {
  const uint32_t plane = (uint32_t)d.nx * (uint32_t)d.ny, slabs = plane / 16384u;
  return slabs > 1u ? ((uint32_t)d.ny + slabs - 1u) / slabs : (uint32_t)d.ny;
}

// Pair e of the level in the order the blocks walk it, so rows narrower than a wave fill
// every lane: slabs of J rows, k planes within a slab, rows within a plane, pairs within a
// row.  False past the last.
__device__ __forceinline__ bool flat_pair(const Dims& d, uint32_t e, uint32_t J, int& p, int& j, int& k) {
  const uint32_t np = (uint32_t)pairs_of(d.nx), ny = (uint32_t)d.ny, nz = (uint32_t)d.nz;
  if (e >= np * ny * nz) return false;
  const uint32_t row = e / np;
  p = (int)(e - row * np);
  if (J >= ny) {
    k = (int)(row / ny);
    j = (int)(row - (uint32_t)k * ny);
    return true;
  }
  const uint32_t j0 = row / (J * nz) * J, in = row - j0 * nz, w = min(J, ny - j0);
  k = (int)(in / w);
  j = (int)(j0 + in - (uint32_t)k * w);
  return true;
}
// cell e of the level, i fastest; false past the last
__device__ __forceinline__ bool flat_cell(const Dims& d, uint32_t e, int& i, int& j, int& k) {
  const uint32_t nxy = (uint32_t)d.nx * (uint32_t)d.ny;
  if (e >= nxy * (uint32_t)d.nz) return false;
  k = (int)(e / nxy);
  const uint32_t r = e - (uint32_t)k * nxy;
  j = (int)(r / (uint32_t)d.nx);
  i = (int)(r - (uint32_t)j * (uint32_t)d.nx);
  return true;
}

// x of another lane of the wave: lane - 1 (CTRL 0x138, wave_shr:1) or lane + 1 (0x130,
// wave_shl:1); `old` where there is no such lane or it is inactive
template <int CTRL, typename T>
__device__ __forceinline__ T lane_shift(T old, T v) {
  if constexpr (sizeof(T) == 8) {
    union U { T d; int i[2]; } a, o;
    a.d = v;
    o.d = old;
    o.i[0] = __builtin_amdgcn_update_dpp(o.i[0], a.i[0], CTRL, 0xF, 0xF, false);
    o.i[1] = __builtin_amdgcn_update_dpp(o.i[1], a.i[1], CTRL, 0xF, 0xF, false);
    return o.d;
  } else if constexpr (sizeof(T) == 4) {
    union U { T f; int i; } a, o;
    a.f = v;
    o.f = old;
    o.i = __builtin_amdgcn_update_dpp(o.i, a.i, CTRL, 0xF, 0xF, false);
    return o.f;
  } else {
    union U { int i; T h[2]; } a, o;
    a.i = o.i = 0;
    a.h[0] = v;
    o.h[0] = old;
    o.i = __builtin_amdgcn_update_dpp(o.i, a.i, CTRL, 0xF, 0xF, false);
    return o.h[0];
  }
}

// Where a pair lies: its first cell's index, the nine stencil rows and the wrapped columns
// beyond it, and which of those the neighbouring lanes hold.  Built by every active lane.
struct PairAt {
  uint32_t c;     // the first cell
  bool both;      // the first cell is this thread's to store
  uint32_t r[9];  // index of column 0 in rows (j, k), (j-1, k), (j+1, k), (j, k-1), (j, k+1),
                  // (j-1, k-1), (j+1, k-1), (j-1, k+1), (j+1, k+1)
  uint32_t i0, im, ip;
  bool in_left, in_right;
};
__device__ __forceinline__ PairAt pair_at(const Dims& d, int p, int j, int k) {
  PairAt q;
  const int i0 = min(2 * p, d.nx - 2);
  const uint32_t sy = (uint32_t)d.nx, sz = (uint32_t)d.nx * (uint32_t)d.ny;
  const uint32_t J = (uint32_t)j * sy, JM = (uint32_t)wrap_m(j, d.ny, d.per[1]) * sy,
                 JP = (uint32_t)wrap_p(j, d.ny, d.per[1]) * sy;
  const uint32_t K = (uint32_t)k * sz, KM = (uint32_t)wrap_m(k, d.nz, d.per[2]) * sz,
                 KP = (uint32_t)wrap_p(k, d.nz, d.per[2]) * sz;
  const uint32_t r[9] = {J + K, JM + K, JP + K, J + KM, J + KP, JM + KM, JP + KM, JM + KP, JP + KP};
#pragma unroll
  for (int s = 0; s < 9; s++) q.r[s] = r[s];
  q.i0 = (uint32_t)i0;
  q.im = (uint32_t)wrap_m(i0, d.nx, d.per[0]);
  q.ip = (uint32_t)wrap_p(i0 + 1, d.nx, d.per[0]);
  q.c = r[0] + (uint32_t)i0;
  q.both = i0 == 2 * p;
  // indices are below 2^29, so no pair's neighbour is taken for one that is missing
  q.in_left = i0 > 0 && lane_shift<0x138>(0x7FFFFFFFu, q.c) + 2u == q.c;
  q.in_right = i0 + 2 < d.nx && lane_shift<0x130>(0x7FFFFFFFu, q.c) == q.c + 2u;
  return q;
}

// x on the stencil of both cells: nine rows of two, and the columns beside the first five
template <typename T>
struct PairX {
  T v[9][2], l[5], r[5];
};
template <typename TX>
__device__ __forceinline__ void pair_load_x(const PairAt& q, const TX* __restrict__ x, PairX<TX>& o) {
#pragma unroll
  for (int s = 0; s < 9; s++) ld_pair(x, q.r[s] + q.i0, o.v[s]);
#pragma unroll
  for (int s = 0; s < 5; s++) o.l[s] = o.r[s] = TX(0);
  if (!q.in_left) {
#pragma unroll
    for (int s = 0; s < 5; s++) o.l[s] = ld_at(x, q.r[s] + q.im);
  }
  if (!q.in_right) {
#pragma unroll
    for (int s = 0; s < 5; s++) o.r[s] = ld_at(x, q.r[s] + q.ip);
  }
}
// the columns the neighbouring lanes hold (after pair_load_x, apart from it so that the
// loads of the coefficients can be issued in between)
template <typename T>
__device__ __forceinline__ void pair_share_x(const PairAt& q, PairX<T>& o) {
#pragma unroll
  for (int s = 0; s < 5; s++) {
    const T l = lane_shift<0x138>(T(0), o.v[s][1]), r = lane_shift<0x130>(T(0), o.v[s][0]);
    o.l[s] = q.in_left ? l : o.l[s];
    o.r[s] = q.in_right ? r : o.r[s];
  }
}

// The coefficients of both rows: own faces, the j-1 and k-1 owners' and the left one's
template <typename TG>
struct PairG {
  TG own[9][2], s[3][2], b[3][2], w[3];
};
template <typename TG>
__device__ __forceinline__ void pair_load_g(const PairAt& q, const TG* __restrict__ g, size_t n, PairG<TG>& o) {
#pragma unroll
  for (int e = 0; e < 9; e++) ld_pair(g + (size_t)e * n, q.c, o.own[e]);
#pragma unroll
  for (int e = 0; e < 3; e++) {
    ld_pair(g + (size_t)(3 + e) * n, q.r[1] + q.i0, o.s[e]);
    ld_pair(g + (size_t)(6 + e) * n, q.r[3] + q.i0, o.b[e]);
    o.w[e] = TG(0);
  }
  if (!q.in_left) {
#pragma unroll
    for (int e = 0; e < 3; e++) o.w[e] = ld_at(g + (size_t)e * n, q.r[0] + q.im);
  }
}
template <typename TG>
__device__ __forceinline__ void pair_share_g(const PairAt& q, PairG<TG>& o) {
#pragma unroll
  for (int e = 0; e < 3; e++) {
    const TG w = lane_shift<0x138>(TG(0), o.own[e][1]);
    o.w[e] = q.in_left ? w : o.w[e];
  }
}

// cell M's stencil values in slot order and its 18 coefficients in face order
template <int M, typename T, typename TX>
__device__ __forceinline__ void pair_xv(const PairX<TX>& x, T (&xv)[19]) {
  const auto e = [&](int s) { return M ? (T)x.r[s] : (T)x.v[s][1]; };
  const auto w = [&](int s) { return M ? (T)x.v[s][0] : (T)x.l[s]; };
  const auto o = [&](int s) { return (T)x.v[s][M]; };
  xv[CP] = o(0), xv[EP] = e(0), xv[WP] = w(0);
  xv[SP] = o(1), xv[SE] = e(1), xv[SW] = w(1);
  xv[NP] = o(2), xv[NE] = e(2), xv[NW] = w(2);
  xv[BP] = o(3), xv[BE] = e(3), xv[BW] = w(3);
  xv[TP] = o(4), xv[TE] = e(4), xv[TW] = w(4);
  xv[BS] = o(5), xv[BN] = o(6), xv[TS] = o(7), xv[TN] = o(8);
}
template <int M, typename TG>
__device__ __forceinline__ void pair_coef(const PairG<TG>& g, RowCoef<TG>& rc) {
#pragma unroll
  for (int e = 0; e < 3; e++) {
    rc.v[0][e] = g.own[e][M];
    rc.v[1][e] = M ? g.own[e][0] : g.w[e];
    rc.v[2][e] = g.own[3 + e][M];
    rc.v[3][e] = g.s[e][M];
    rc.v[4][e] = g.own[6 + e][M];
    rc.v[5][e] = g.b[e][M];
  }
}
template <int KC, typename T, typename TG, typename TX>
__device__ __forceinline__ void pair_flux(const PairG<TG>& g, const PairX<TX>& x, const uint32_t (&code)[2],
                                          T (&ax)[2], T (&dg)[2]) {
  RowCoef<TG> rc;
  T xv[19];
  pair_xv<0>(x, xv);
  pair_coef<0>(g, rc);
  flux_row_v<KC>(rc, code[0], xv, ax[0], dg[0]);
  pair_xv<1>(x, xv);
  pair_coef<1>(g, rc);
  flux_row_v<KC>(rc, code[1], xv, ax[1], dg[1]);
}

// (A x) on both cells, each row in the form its wave takes (see flux_row)
template <typename TG, typename TX, typename T>
__device__ __forceinline__ void pair_apply(const PairAt& q, const TG* __restrict__ g, size_t n,
                                           const uint32_t* __restrict__ code, const TX* __restrict__ x,
                                           uint32_t (&cd)[2], PairX<TX>& xs, T (&ax)[2], T (&dg)[2]) {
  PairG<TG> gs;
  ld_pair(code, q.c, cd);
  pair_load_x(q, x, xs);
  pair_load_g(q, g, n, gs);
  pair_share_x(q, xs);
  pair_share_g(q, gs);
  if (__all((cd[0] & ~DIVOK_BIT) == CODE_INTERIOR && (cd[1] & ~DIVOK_BIT) == CODE_INTERIOR))
    pair_flux<X_CENTRAL>(gs, xs, cd, ax, dg);
  else
    pair_flux<-1>(gs, xs, cd, ax, dg);
}

}  // namespace pp
