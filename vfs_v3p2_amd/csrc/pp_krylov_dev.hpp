// Device bodies of the FGMRES basis kernels (classical Gram-Schmidt with
// re-orthogonalisation, fused into three passes over the basis).  Shared by the
// single-case kernels (pp_core.hip) and the batched kernels (pp_batch.hip).
#pragma once

#include "pp_common.hpp"
#include "pp_pair_dev.hpp"
#include "pp_stencil.hpp"

namespace pp {

// Per-block sums of a * V_l[c] for l < nv and of a * a (slot nv), written to
// partial[l * nblk + b].  Eight vectors at a time are loaded together, reduced
// inside each wave by shuffles and parked in LDS; one barrier, then thread l
// adds the four wave sums of slot l.  256-thread blocks, nv < 64; every thread
// of the block must call it.
__device__ inline void block_dots(bool in, size_t c, double a, const double* __restrict__ V, size_t ldv, int nv,
                                  double* __restrict__ partial, size_t nblk, size_t b, double (*lds)[64]) {
  const int t = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  const int lane = t & 63, w = t >> 6;
  for (int l0 = 0; l0 <= nv; l0 += 8) {
    double p[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int l = l0 + q;
      double v = 0.;
      if (in && l < nv) v = a * V[(size_t)l * ldv + c];
      else if (in && l == nv) v = a * a;
      p[q] = v;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) p[q] = wave_sum(p[q]);
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (l0 + q <= nv) lds[w][l0 + q] = p[q];
    }
  }
  __syncthreads();
  if (t <= nv) partial[(size_t)t * nblk + b] = (lds[0][t] + lds[1][t]) + (lds[2][t] + lds[3][t]);
  __syncthreads();  // lds is reused by the block's next tile
}

// x from a lane DPP_CTRL selects (0 where the source lane is out of its row or
// the lane is masked out by row_mask / bank_mask), a double moved as two dwords
template <int DPP_CTRL, int ROW_MASK, int BANK_MASK>
__device__ __forceinline__ double dpp_f64(double x) {
  union {
    double d;
    int i[2];
  } u, r;
  u.d = x;
  r.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], DPP_CTRL, ROW_MASK, BANK_MASK, true);
  r.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], DPP_CTRL, ROW_MASK, BANK_MASK, true);
  return r.d;
}

// Sum of v over the 64 lanes of a wave, left in lane 63 (other lanes hold partial
// sums), without LDS: row shifts by 1, 2, 4 and 8 leave each row's sum in its
// last lane, then row broadcasts 15 and 31 carry the row sums into lane 63.
// Every lane of the wave must be active.
__device__ __forceinline__ double wave_sum_to63(double v) {
  v += dpp_f64<0x111, 0xF, 0xF>(v);  // row_shr:1
  v += dpp_f64<0x112, 0xF, 0xF>(v);  // row_shr:2
  v += dpp_f64<0x114, 0xF, 0xE>(v);  // row_shr:4 into banks 1-3
  v += dpp_f64<0x118, 0xF, 0xC>(v);  // row_shr:8 into banks 2-3
  v += dpp_f64<0x142, 0xA, 0xF>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_f64<0x143, 0xC, 0xF>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// V_l on the N cells from c for l < min(nv, DOTS_AHEAD), loaded before the values they
// multiply are computed so the loads overlap that computation
constexpr int DOTS_AHEAD = 4;
template <int N>
__device__ __forceinline__ void wave_dots_prefetch(bool in, uint32_t c, const double* __restrict__ V, size_t ldv,
                                                   int nv, double (&va)[DOTS_AHEAD][N]) {
#pragma unroll
  for (int q = 0; q < DOTS_AHEAD; q++) {
#pragma unroll
    for (int m = 0; m < N; m++) va[q][m] = 0.;
    if (in && q < nv) {
      if constexpr (N == 2) ld_pair(V + (size_t)q * ldv, c, va[q]);
      else va[q][0] = ld_at(V + (size_t)q * ldv, c);
    }
  }
}

// Per-wave sums of a . V_l over each thread's N cells for l < nv and of a . a (slot nv),
// written by the wave's last lane to partial[l * nw + wv] (nw waves in the launch, wv this
// wave's index).  c is the first cell; a is 0 where a cell is another thread's.  va holds
// the first DOTS_AHEAD vectors (wave_dots_prefetch); the rest are loaded as many at a time.
// Every lane of the wave must call it (cells outside the grid pass in = false); nv < 64.
template <int N>
__device__ inline void wave_dots(bool in, uint32_t c, const double (&a)[N], const double* __restrict__ V, size_t ldv,
                                 int nv, double (&va)[DOTS_AHEAD][N], double* __restrict__ partial, size_t nw,
                                 size_t wv) {
  const int lane = (threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z)) & 63;
  double own = 0.;
#pragma unroll
  for (int m = 0; m < N; m++) own += a[m] * a[m];
  own = wave_sum_to63(in ? own : 0.);
  if (lane == 63) partial[(size_t)nv * nw + wv] = own;
  for (int l0 = 0; l0 < nv; l0 += DOTS_AHEAD) {
    if (l0 > 0) wave_dots_prefetch(in, c, V + (size_t)l0 * ldv, ldv, nv - l0, va);
    double p[DOTS_AHEAD];
#pragma unroll
    for (int q = 0; q < DOTS_AHEAD; q++) {
      p[q] = 0.;
#pragma unroll
      for (int m = 0; m < N; m++) p[q] += a[m] * va[q][m];
      p[q] = wave_sum_to63(in ? p[q] : 0.);
    }
    if (lane == 63) {
#pragma unroll
      for (int q = 0; q < DOTS_AHEAD; q++)
        if (l0 + q < nv) partial[(size_t)(l0 + q) * nw + wv] = p[q];
    }
  }
}

// Per-block sums of per-thread accumulators acc[0..ns) (ns <= S <= 64), written to
// partial[l * nblk + b]: wave sums by shuffles, the four wave results of a
// 256-thread block meet in LDS.  Every thread of the block must call it.
template <int S>
__device__ inline void block_sums(const double (&acc)[S], int ns, double* __restrict__ partial, size_t nblk,
                                  size_t b, double (*lds)[64]) {
  const int t = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  const int lane = t & 63, w = t >> 6;
#pragma unroll
  for (int l = 0; l < S; l++) {
    if (l < ns) {
      const double v = wave_sum(acc[l]);
      if (lane == 0) lds[w][l] = v;
    }
  }
  __syncthreads();
  if (t < ns) partial[(size_t)t * nblk + b] = (lds[0][t] + lds[1][t]) + (lds[2][t] + lds[3][t]);
  __syncthreads();  // lds is reused by the block's next call
}

// gs_sub followed by block_dots of the result at element t, with the basis
// values V_l[t] (l < nv <= S) loaded once into registers for both; the same
// arithmetic as the two calls.  Every thread of the block must call it.
template <int S>
__device__ inline void gs_sub_block_dots(bool in, double* __restrict__ w, const double* __restrict__ V, size_t ldv,
                                         int nv, const double* __restrict__ h, size_t t,
                                         double* __restrict__ partial, size_t nblk, size_t b, double (*lds)[64]) {
  const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  const int lane = tid & 63, wv = tid >> 6;
  double vv[S];
#pragma unroll
  for (int l = 0; l < S; l++) vv[l] = (in && l < nv) ? V[(size_t)l * ldv + t] : 0.;
  double w1 = 0.;
  if (in) {
    w1 = w[t];
#pragma unroll
    for (int l = 0; l < S; l++)
      if (l < nv) w1 -= h[l] * vv[l];
    w[t] = w1;
  }
#pragma unroll
  for (int l0 = 0; l0 <= S; l0 += 8) {
    if (l0 > nv) break;
    double p[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int l = l0 + q;
      double v = 0.;
      if (in && l < nv && l < S) v = w1 * vv[l < S ? l : 0];
      else if (in && l == nv) v = w1 * w1;
      p[q] = v;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) p[q] = wave_sum(p[q]);
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (l0 + q <= nv) lds[wv][l0 + q] = p[q];
    }
  }
  __syncthreads();
  if (tid <= nv) partial[(size_t)tid * nblk + b] = (lds[0][tid] + lds[1][tid]) + (lds[2][tid] + lds[3][tid]);
  __syncthreads();  // lds is reused by the block's next tile
}

// Power of two near 1/||w|| from ||w||^2, the scale of the single-precision copy
// of an unnormalised basis vector (the host computes the same value).
__host__ __device__ inline double conv_scale(double a2) {
  if (!(a2 > 0.)) return 1.;
  const int e = ilogb(a2);
  return ldexp(1.0, -(int)floor(0.5 * e));
}

// w = A z in flux form on the pair's row cells, 0 elsewhere; wv: w, 0 on a first cell that
// is another thread's
template <typename TZ>
__device__ __forceinline__ void apply_pair(const Dims& d, const PairAt& at, const double* __restrict__ g,
                                           const uint32_t* __restrict__ code, const TZ* __restrict__ z,
                                           double* __restrict__ w, double (&wv)[2]) {
  uint32_t cd[2];
  PairX<TZ> xs;
  double ax[2], dg[2];
  pair_apply(at, g, d.n(), code, z, cd, xs, ax, dg);
  const double w0 = (cd[0] & ROW_BIT) ? ax[0] : 0.;
  wv[1] = (cd[1] & ROW_BIT) ? ax[1] : 0.;
  wv[0] = at.both ? w0 : 0.;
  st_pair(w, at.c, at.both, w0, wv[1]);
}

// the same on one cell
template <typename TZ>
__device__ __forceinline__ double apply_cell(const Dims& d, const double* __restrict__ g,
                                             const uint32_t* __restrict__ code, const TZ* __restrict__ z,
                                             double* __restrict__ w, int i, int j, int k) {
  const size_t c = d.idx(i, j, k);
  const uint32_t cd = code[c];
  Nbr nb;
  neighbours(d, i, j, k, nb);
  double xv[19], ax, dg;
  load_x(nb, z, xv);
  flux_row(g, d.n(), cd, c, nb.s[WP], nb.s[SP], nb.s[BP], xv, ax, dg);
  const double wv = (cd & ROW_BIT) ? ax : 0.;
  w[c] = wv;
  return wv;
}

// w = A z on the cells of thread e (pairs: a flat walk of pairs, else of cells) and the
// wave's partial sums of w.V_l (l < nv) and w.w; e is past the last on idle threads.
template <bool PAIRS, typename TZ>
__device__ __forceinline__ void apply_dots(const Dims& d, uint32_t slab, uint32_t e, const double* __restrict__ g,
                                           const uint32_t* __restrict__ code, const TZ* __restrict__ z,
                                           double* __restrict__ w, const double* __restrict__ V, size_t ldv, int nv,
                                           double* __restrict__ partial, size_t nw, size_t wave) {
  int i = 0, j = 0, k = 0;
  if constexpr (PAIRS) {
    const bool in = flat_pair(d, e, slab, i, j, k);
    double va[DOTS_AHEAD][2], wv[2] = {0., 0.};
    PairAt at{};
    if (in) at = pair_at(d, i, j, k);
    wave_dots_prefetch(in, at.c, V, ldv, nv, va);
    if (in) apply_pair(d, at, g, code, z, w, wv);
    wave_dots(in, at.c, wv, V, ldv, nv, va, partial, nw, wave);
  } else {
    const bool in = flat_cell(d, e, i, j, k);
    const uint32_t c = in ? (uint32_t)d.idx(i, j, k) : 0u;
    double va[DOTS_AHEAD][1], wv[1] = {0.};
    wave_dots_prefetch(in, c, V, ldv, nv, va);
    if (in) wv[0] = apply_cell(d, g, code, z, w, i, j, k);
    wave_dots(in, c, wv, V, ldv, nv, va, partial, nw, wave);
  }
}

// The lazily normalised Gram-Schmidt update on the elements 2t and 2t + 1 (of an odd n the
// last thread's pair overlaps the one before and stores its second element only):
// w' = w - sum_l (dots_l nuinv2_l) V_l in place, f = (T)(w' sc).  Four vectors' pairs are
// loaded at a time, so a thread waits for memory once per four vectors instead of once per
// vector and element.  Returns |w'|^2 over the elements stored.
template <typename T>
__device__ __forceinline__ double axpy_norm_pair(uint32_t t, uint32_t n, double* __restrict__ w,
                                                 const double* __restrict__ V, size_t ldv, int nv,
                                                 const double* __restrict__ dots, const double* __restrict__ nuinv2,
                                                 double sc, T* __restrict__ f) {
  const uint32_t e = min(2 * t, n - 2);
  const bool both = e == 2 * t;
  double va[DOTS_AHEAD][2], v[2];
  ld_pair((const double*)w, e, v);
  for (int l0 = 0; l0 < nv; l0 += DOTS_AHEAD) {
    wave_dots_prefetch(true, e, V + (size_t)l0 * ldv, ldv, nv - l0, va);
#pragma unroll
    for (int q = 0; q < DOTS_AHEAD; q++)
      if (l0 + q < nv) {
        const double c = dots[l0 + q] * nuinv2[l0 + q];
        v[0] -= c * va[q][0];
        v[1] -= c * va[q][1];
      }
  }
  st_pair(w, e, both, v[0], v[1]);
  st_pair(f, e, both, (T)(v[0] * sc), (T)(v[1] * sc));
  return (both ? v[0] * v[0] : 0.) + v[1] * v[1];
}

// w1 = w - sum_l h_l V_l at element t (in place); returns w1
__device__ __forceinline__ double gs_sub(double* __restrict__ w, const double* __restrict__ V, size_t ldv, int nv,
                                         const double* __restrict__ h, size_t t) {
  double w1 = w[t];
  for (int l = 0; l < nv; l++) w1 -= h[l] * V[(size_t)l * ldv + t];
  w[t] = w1;
  return w1;
}

// red[1] = ||w - V h|| = sqrt(w.w - h.h), red[2] = 1/red[1] with h = red[off..off+nv)
// and w.w = red[off+nv]; mirrored to host.  One thread.
__device__ __forceinline__ void gs_norm_one(double* __restrict__ red, int off, int nv, double* __restrict__ host) {
  const double* h = red + off;
  double hh = 0.;
  for (int l = 0; l < nv; l++) hh += h[l] * h[l];
  const double s = h[nv] - hh;  // h[nv] holds w.w
  const double nrm = s > 0. ? sqrt(s) : 0.;
  red[1] = nrm;
  red[2] = nrm > 0. ? 1. / nrm : 0.;
  if (host) { host[1] = nrm; host[2] = red[2]; }
}

// v = (w - sum_l h_l V_l) * inv at element t (in place over w); f = (TF)v
template <typename TF>
__device__ __forceinline__ void axpy_scale_one(double* __restrict__ w, const double* __restrict__ V, size_t ldv,
                                               int nv, const double* __restrict__ h, double inv, TF* __restrict__ f,
                                               size_t t) {
  double acc = w[t];
  for (int l = 0; l < nv; l++) acc -= h[l] * V[(size_t)l * ldv + t];
  const double v = acc * inv;
  w[t] = v;
  if (f) f[t] = (TF)v;
}

}  // namespace pp
