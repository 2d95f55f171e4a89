// Pressure_Gradient (momentum.c:223-452) on the device: the contravariant
// pressure-gradient flux dP on the i, j and k faces of every interior cell from P
// and the face metrics, for the momentum step that follows the projection.
// Levelset density, the -dpdz mean-gradient forcing and the -flux inlet
// correction are off, as they are by default (main.c:73, 95).  The arithmetic
// keeps the reference's operand order and the kernel is compiled without
// contraction, so dP is bit-exact with a CPU restatement.
#include "pp_engine.hpp"

namespace pp {

namespace {

#pragma clang fp contract(off)

struct GradIn {
  const double *icsi, *ieta, *izet, *jcsi, *jeta, *jzet, *kcsi, *keta, *kzet, *iaj, *jaj, *kaj, *nvert;
};

__device__ __forceinline__ double dot3(const double* a, const double* b, size_t c) {
  return a[3 * c] * b[3 * c] + a[3 * c + 1] * b[3 * c + 1] + a[3 * c + 2] * b[3 * c + 2];
}

// One thread per DMDA point, 256 consecutive points per block, blocks in XCD order.  P at the 19 points the three faces'
// differences may read (and the periodic ones beyond the last cell) and the masks beside
// them are loaded before any case is decided, so a point waits for memory once instead of
// once per branch (192x96x128: 269 -> 161 us).
__global__ __launch_bounds__(256) void k_pressure_gradient(Dmda m, GradIn in, const double* __restrict__ p,
                                                           double* __restrict__ dp) {
  const uint32_t c = xcd_block().x * 256u + threadIdx.x, mxy = (uint32_t)m.mx * (uint32_t)m.my;
  if (c >= mxy * (uint32_t)m.mz) return;
  const int k = (int)(c / mxy), j = (int)((c - (uint32_t)k * mxy) / (uint32_t)m.mx);
  const int i = (int)(c - (uint32_t)k * mxy - (uint32_t)j * (uint32_t)m.mx);
  if (i == 0 || j == 0 || k == 0 || i == m.mx - 1 || j == m.my - 1 || k == m.mz - 1) {
    dp[3 * c] = 0.;  // VecSet(dP, 0.): only interior points are written below
    dp[3 * c + 1] = 0.;
    dp[3 * c + 2] = 0.;
    return;
  }
  const int pos[3] = {i, j, k}, mm[3] = {m.mx, m.my, m.mz};
  const size_t st[3] = {1, (size_t)m.mx, (size_t)m.mx * m.my};
  const double p0 = p[c];
  double ph[3], pl[3], pw[3];        // +a, -a, and the +a point across a periodic end
  double phh[3][3], phl[3][3];       // [a][e]: +a +e and +a -e, e != a (phh symmetric)
  double nh[3], nl[3], nhh[3][3], nhl[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    ph[a] = p[c + st[a]];
    pl[a] = p[c - st[a]];
    pw[a] = (pos[a] == mm[a] - 2 && m.per[a]) ? p[c - (size_t)(pos[a] - 1) * st[a]] : ph[a];
    nh[a] = in.nvert[c + st[a]];
    nl[a] = in.nvert[c - st[a]];
  }
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int e = 0; e < 3; e++) {
      if (e == a) continue;
      phl[a][e] = p[c + st[a] - st[e]];
      nhl[a][e] = in.nvert[c + st[a] - st[e]];
      if (a < e) {
        phh[a][e] = phh[e][a] = p[c + st[a] + st[e]];
        nhh[a][e] = nhh[e][a] = in.nvert[c + st[a] + st[e]];
      }
    }
  const double g[3][3] = {{dot3(in.icsi, in.icsi, c), dot3(in.ieta, in.icsi, c), dot3(in.izet, in.icsi, c)},
                          {dot3(in.jcsi, in.jeta, c), dot3(in.jeta, in.jeta, c), dot3(in.jzet, in.jeta, c)},
                          {dot3(in.kcsi, in.kzet, c), dot3(in.keta, in.kzet, c), dot3(in.kzet, in.kzet, c)}};
  const double aj[3] = {in.iaj[c], in.jaj[c], in.kaj[c]};
  const double nv = in.nvert[c];
  auto N1 = [](double v) { return (int)(v + 0.5) == 1; };
  // face a (momentum.c:352-364, 366-380, 382-396): the difference across it, and along each
  // other axis e the pair sums of the two cells beside the face, one-sided next to nvert 1
  // cells and non-periodic walls
#pragma unroll
  for (int a = 0; a < 3; a++) {
    double d[3];
#pragma unroll
    for (int e = 0; e < 3; e++) {
      if (e == a) {
        d[e] = pw[a] - p0;
      } else {
        const bool hi = N1(nh[e]) || N1(nhh[a][e]) || (pos[e] == mm[e] - 2 && !m.per[e]);
        const bool lo = !hi && (N1(nl[e]) || N1(nhl[a][e]) || (pos[e] == 1 && !m.per[e]));
        const double u0 = hi ? p0 : ph[e], u1 = hi ? ph[a] : phh[a][e];
        const double l0 = lo ? p0 : pl[e], l1 = lo ? ph[a] : phl[a][e];
        d[e] = (u0 - l0 + u1 - l1) * (hi || lo ? 0.5 : 0.25);
      }
    }
    double f = (d[0] * g[a][0] + d[1] * g[a][1] + d[2] * g[a][2]) * aj[a];
    // faces without a fluid pair or on a non-periodic wall carry none (momentum.c:426-436)
    if (nv + nh[a] > 0.1 || (!m.per[a] && pos[a] == mm[a] - 2)) f = 0;
    dp[3 * c + a] = f;
  }
}

}  // namespace

}  // namespace pp

using namespace pp;

int vfs_pp_pressure_gradient_device(const vfs_grid* g, const double* icsi, const double* ieta, const double* izet,
                                    const double* jcsi, const double* jeta, const double* jzet, const double* kcsi,
                                    const double* keta, const double* kzet, const double* iaj, const double* jaj,
                                    const double* kaj, const double* nvert, double* p, double* dp) {
  ABI_BEGIN
  if (!g || !nvert || !p || !dp) return VFS_PP_EINVAL;
  const double* mt[12] = {icsi, ieta, izet, jcsi, jeta, jzet, kcsi, keta, kzet, iaj, jaj, kaj};
  for (auto q : mt)
    if (!q) return VFS_PP_EINVAL;
  if (g->nx < 2 || g->ny < 2 || g->nz < 2) return VFS_PP_EINVAL;
  const Dmda m{g->nx + 2, g->ny + 2, g->nz + 2, {g->periodic[0] ? 1 : 0, g->periodic[1] ? 1 : 0, g->periodic[2] ? 1 : 0}};
  // periodic ghost copies of P (momentum.c:270-307), then the face fluxes
  launch_periodic_scalar(nullptr, m, p, 0);
  const GradIn in{icsi, ieta, izet, jcsi, jeta, jzet, kcsi, keta, kzet, iaj, jaj, kaj, nvert};
  k_pressure_gradient<<<(unsigned)((m.n() + 255) / 256), 256, 0, nullptr>>>(m, in, p, dp);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipDeviceSynchronize());
  return VFS_PP_OK;
  ABI_END
}
