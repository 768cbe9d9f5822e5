// qas_common.hip -- boundary fill and CFL reduction kernels (all dimensions).
//
//   k_bound     bound(val) = bc1d / bc2d / bc3d (common/common_func.c:34-278)
//               on one device-resident domain: each ghost cell is written
//               once from the kept cell that the x -> y -> z passes of the
//               reference would copy into it, times the pass factors.
//   k_cfl       setdt(1)'s max of |v| + vfast over the interior with the
//               2nd-order cell-centred B (mhd2d_class.cpp:11-33,
//               mhd1d_class.cpp:11-30, mhd3d_class.cpp:15-46): grid-stride
//               loop, wavefront max by cross-lane shuffles, block max in
//               LDS, one partial maximum per block (no atomics).
//   k_cfl_final dt = cfl*dr/vmax into device memory from the partials,
//               with the reference's floor vmax >= 1.0.
#include "qas_common.hpp"
#include "qas_device.hpp"
#include "qas_internal.hpp"

namespace qas {

__global__ __launch_bounds__(256) void k_bound(BoundArgs a, Geo g, BcFlags bc, long long nghost, int ox, int oy,
                                               int oz)
{
  bound_at_f([&](int m) { return a.f[m]; }, a.nvar, a.phi, a.gfac, g, bc, nghost, ox, oy, oz,
             (long long)blockIdx.x * blockDim.x + threadIdx.x);
}

// 3D: every variable of a ghost cell per thread, so that a cell is located
// once for all eight and the eight copies are in flight together (a variable
// per thread, located with 64-bit divisions: 29.2 us at 128^3, 74 at 200^3;
// this form 20 and 50)
__global__ __launch_bounds__(256) void k_bound3(BoundArgs a, Geo g, BcFlags bc, unsigned nghost)
{
  const unsigned r = blockIdx.x * 256u + threadIdx.x;
  if (r >= nghost) return;
  int i, j, k;
  ghost_cell(g, NG, NG, NG, r, i, j, k);
  bool keep[8];
  double v[8];
#pragma unroll
  for (int m = 0; m < 8; m++) {
    if (m >= a.nvar) break;
    const Src sx = resolve(i, g.nx, bc.st[0][m], bc.dn[0][m]);
    const Src sy = resolve(j, g.ny, bc.st[1][m], bc.dn[1][m]);
    const Src sz = resolve(k, g.nz, bc.st[2][m], bc.dn[2][m]);
    keep[m] = sx.i == i && sy.i == j && sz.i == k;  // (staggered boundary face)
    v[m] = apply(sz, apply(sy, apply(sx, a.f[m][g.sz * sz.i + g.sy * sy.i + sx.i])));
  }
  const long long s = g.sz * k + g.sy * j + i;
#pragma unroll
  for (int m = 0; m < 8; m++) {
    if (m >= a.nvar) break;
    if (!keep[m]) a.f[m][s] = v[m];
  }
}

hipError_t launch_bound(qas_ctx* c, double* const f[8], int nvar)
{
  const Geo& g = c->geo;
  const int ox = qas::NG;
  const int oy = g.ndim >= 2 ? qas::NG : 0;
  const int oz = g.ndim >= 3 ? qas::NG : 0;
  const long long nghost = (long long)g.nx * g.ny * g.nz -
                           (long long)(g.nx - 2 * ox) * (g.ny - 2 * oy) * (g.nz - 2 * oz);
  BoundArgs a;
  for (int m = 0; m < 8; m++) a.f[m] = f[m];
  a.nvar = nvar;
  if (c->d_phi && nvar == 8) {
    a.phi = c->d_phi;
    a.gfac = (2.0 - c->s.gam) / (c->s.gam - 1.0);
  }
  if (g.ndim == 3) {
    QAS_LAUNCH(c, QAS_K_BOUND, k_bound3, (unsigned)((nghost + 255) / 256), 256, 0, c->stream, a, g, c->bc,
               (unsigned)nghost);
    return hipGetLastError();
  }
  const long long tot = nghost * nvar;
  QAS_LAUNCH(c, QAS_K_BOUND, k_bound, (unsigned)((tot + 255) / 256), 256, 0, c->stream, a, g, c->bc, nghost, ox, oy, oz);
  return hipGetLastError();
}

// ------------------------------------------------------------------ CFL
__global__ __launch_bounds__(256) void k_cfl(CflArgs a, Geo g) { cfl_block(a, g, (int)blockIdx.x, (int)gridDim.x); }

// A small domain's whole reduction in one workgroup of 1024 threads, one cell
// each: 3.9 us at 1024 cells against 3.8 + 3.8 for two launches.  With 4 cells
// per thread (64^2) it took 10.0 us against 4.2 + 3.8.
constexpr long long CFL_ONE = 1024;
__global__ __launch_bounds__(1024) void k_cfl_one(CflArgs a, Geo g, double* dt, double cfl_dr)
{
  __shared__ double wm[16];
  double v = wave_max(cfl_thread(a, g, 0, 1));
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; w++) v = (wm[w] > v) ? wm[w] : v;
    *dt = cfl_dr / v;
  }
}

__global__ __launch_bounds__(256) void k_cfl_final(const double* part, int nb, double* dt, double cfl_dr)
{
  cfl_final_block(part, nb, dt, cfl_dr);
}

__global__ void k_set_dt(double* dt, double v) { *dt = v; }
// dt history for graph replays: hist[*cnt] = *dt; ++*cnt (one thread)
__global__ void k_record(const double* dt, double* hist, long long* cnt, long long cap)
{
  const long long n = *cnt;
  if (n < cap) hist[n] = *dt;
  *cnt = n + 1;
}

// the smallest cell size of the active axes
static double cell_size(const Geo& g)
{
  double dr = g.dx;
  if (g.ndim == 2) dr = (g.dx >= g.dy) ? g.dy : g.dx;
  if (g.ndim == 3) {
    const double t = (g.dx >= g.dy) ? g.dy : g.dx;
    dr = (t >= g.dz) ? g.dz : t;
  }
  return dr;
}

hipError_t launch_cfl(qas_ctx* c, const double* const U[8])
{
  const Geo& g = c->geo;
  CflArgs a;
  for (int m = 0; m < 8; m++) a.u[m] = U[m];
  a.part = c->d_cflpart;
  a.gam = c->s.gam;
  a.stx4 = c->s.st[0][4];
  a.sty5 = c->s.st[1][5];
  a.stz6 = c->s.st[2][6];
  if (c->d_phi) {
    a.phi = c->d_phi;
    a.enw = const_cast<double*>(U[7]);
    c->bounded = false;  // the interior energy is rewritten: its ghosts are stale
  }
  const int ox = qas::NG, oy = g.ndim >= 2 ? qas::NG : 0, oz = g.ndim >= 3 ? qas::NG : 0;
  const long long n = (long long)(g.nx - 2 * ox) * (g.ny - 2 * oy) * (g.nz - 2 * oz);
  if (n <= CFL_ONE) {
    c->cfl_blocks = 0;
    QAS_LAUNCH(c, QAS_K_CFL, k_cfl_one, 1, 1024, 0, c->stream, a, g, c->d_dt, c->s.cfl * cell_size(g));
    return hipGetLastError();
  }
  long long nb = (n + 255) / 256;
  if (nb > CFL_MAX_BLOCKS) nb = CFL_MAX_BLOCKS;
  c->cfl_blocks = (int)nb;
  QAS_LAUNCH(c, QAS_K_CFL, k_cfl, (unsigned)nb, 256, 0, c->stream, a, g);
  return hipGetLastError();
}

hipError_t launch_cfl_finalize(qas_ctx* c)
{
  if (c->cfl_blocks == 0) return hipGetLastError();  // k_cfl_one has set dt
  const double cfl_dr = c->s.cfl * cell_size(c->geo);
  hipLaunchKernelGGL(k_cfl_final, 1, 256, 0, c->stream, c->d_cflpart, c->cfl_blocks, c->d_dt, cfl_dr);
  return hipGetLastError();
}

hipError_t launch_set_dt(qas_ctx* c, double dt)
{
  hipLaunchKernelGGL(k_set_dt, 1, 1, 0, c->stream, c->d_dt, dt);
  return hipGetLastError();
}

hipError_t launch_record_counted(qas_ctx* c)
{
  hipLaunchKernelGGL(k_record, 1, 1, 0, c->stream, c->d_dt, c->d_hist, c->d_hcount, (long long)c->hist_cap);
  return hipGetLastError();
}

__global__ void k_zero_ll(long long* p) { *p = 0; }

hipError_t launch_zero_counter(qas_ctx* c)
{
  hipLaunchKernelGGL(k_zero_ll, 1, 1, 0, c->stream, c->d_hcount);
  return hipGetLastError();
}

}  // namespace qas
