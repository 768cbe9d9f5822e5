// qas_kernels3d.hip -- one SSP-RK stage of the 3D ideal-MHD step on gfx950.
//
// Replaces the stage body of MHD3D::ideal (3D/MPI/OTvortex/mhd3d_solve.cpp:
// 42-715) on one device-resident domain:
//   sweep<d>  for d = z, y, x: characteristic WCNS + Riemann flux on every
//             line; z and y store dt/dz Dz and dt/dy Dy of ro, mx, my, mz,
//             en, the x sweep applies the RK stage sum with the reference's
//             ((-dtdx Dx) - dtdy Dy) - dtdz Dz; upwind/central parts of both
//             tangential B fluxes stored per face          (:166-258, 330-422, 494-586, 658-676);
//             the z sweep first computes the cell-centred B (fcen along x,
//             y, z; ghosts by the bound() index map) and primitives of its
//             LDS tile and stores them for the y and x sweeps (:49-98)
//   emf3d     Ex, Ey, Ez at cell edges from the face parts (CUCT)
//                                                            (:100-136, 259-328, 423-492, 587-656)
//   ct3d      staggered bx, by, bz update                    (:677-709)
// followed by the bound() kernel (:713-714).
#include "qas_device.hpp"
#include "qas_internal.hpp"
#include "qas_sweep3d.hpp"

namespace qas {

// the face sweeps live in qas_sweep3d.hpp (shared with the mixed path)

// ------------------------------------------------------------------ EMF
// Edge EMFs Ex, Ey, Ez (CUCT, mhd3d_solve.cpp:100-136, 259-328, 423-492,
// 587-656).  Each component is two interpolations of a sweep's face parts
// (upwind fu, central fc) to the edge, along the edge's two transverse axes,
//   sgn ((uL + uR) + w (cL + cR)),
// weighted with the CUCT weight of the four cells around it.  A thread forms
// one component at a row of edges along one of those axes (z for Ex and Ey, y
// for Ez): the parts interpolated along it sit in 6-point register windows and
// the two cells behind are carried, so each is read once.  Per edge the
// operations and their order are the reference's.
// One thread for all three components takes 256 VGPRs (2 wavefronts per SIMD)
// and waits on its loads where there are few columns: 182 us at 128^3 (FP64),
// 383 at 200^3 (mixed); one component per thread 147 and 336 (116 VGPRs).
// Large domains: k_emf3d_z.
// FT: the sweep precision, the type of the face parts, of the velocities (the
// primitives the z sweep stored) and of the edge EMFs; arithmetic is FP64.
template <int ODR>
__device__ __forceinline__ double emf_part_w(const double (&u)[6], const double (&c)[6], double w, double sgn)
{
  double a[5], b[5], ul0, ur0, ul1, ur1, dum;
#pragma unroll
  for (int m = 0; m < 5; m++) { a[m] = u[m]; b[m] = c[m]; }
  lin5<ODR>(a, ul0, dum);
  lin5<ODR>(b, ul1, dum);
#pragma unroll
  for (int m = 0; m < 5; m++) { a[m] = u[m + 1]; b[m] = c[m + 1]; }
  lin5<ODR>(a, dum, ur0);
  lin5<ODR>(b, dum, ur1);
  return sgn * ((ul0 + ur0) + w * (ul1 + ur1));
}

// component E (0 x, 1 y, 2 z) at the edges of one row: q counts the edges of
// the plane (x, the axis that is not marched), chunk the runs of kc edges
template <int E, int ODR, typename FT>
__device__ __forceinline__ void emf3d_row(const StagePtrs& p, const Geo& g, int ctw, unsigned q, int chunk, int kc)
{
  constexpr int XA = (E + 1) % 3, YA = (E + 2) % 3;  // cuct_weight's axes (xo, yo)
  constexpr int MA = E == 2 ? 1 : 2;                 // marched axis
  constexpr int OA = E == 2 ? 2 : (E == 0 ? 1 : 1);  // the plane's other axis besides x
  constexpr bool MY = MA == YA;                      // marching along yo (Ex, Ez) or xo (Ey)
  constexpr int IA = MY ? XA : YA;                   // the other interpolation axis
  const int dims[3] = {g.nx, g.ny, g.nz};
  const long long strd[3] = {1, g.sy, g.sz};
  const unsigned ni = (unsigned)g.nx - 5;            // edges on [3, n-3]
  const unsigned row = q / ni;
  if (row >= (unsigned)dims[OA] - 5) return;
  const int i = 3 + (int)(q - row * ni), j = 3 + (int)row;
  const int k0 = 3 + chunk * kc, n = dims[MA];
  const int k1 = k0 + kc < n - 2 ? k0 + kc : n - 2;
  const long long sm = strd[MA], si = strd[IA];
  long long ss = sm * k0 + strd[OA] * j + i;
  // face parts: along the marched axis, and along the other one
  constexpr int PM = E == 0 ? 4 : (E == 1 ? 2 : 0), PI = E == 0 ? 10 : (E == 1 ? 8 : 6);
  constexpr double SM = E == 1 ? 0.5 : -0.5, SI = -SM;
  const double *ro = p.in[0], *ba = p.in[4 + XA], *bb = p.in[4 + YA];
  const double* const vel[3] = {p.vx, p.vy, p.vz};
  const double *va = vel[XA], *vb = vel[YA];
  double u[6], c[6];
#pragma unroll
  for (int m = 0; m < 5; m++) {
    u[m] = load_as<FT>(p.emf[PM], ss + (m - 3) * sm);
    c[m] = load_as<FT>(p.emf[PM + 1], ss + (m - 3) * sm);
  }
  // the cells behind along the marched axis: at the edge's row and one back
  // along the other axis
  double rb0 = 0, rb1 = 0, ab0 = 0, ab1 = 0, cb0 = 0, cb1 = 0, fb = 0;
  if (ctw) {
    const long long s = ss - sm;
    rb0 = ro[s]; rb1 = ro[s - si];
    ab0 = load_as<FT>(va, s); ab1 = load_as<FT>(va, s - si);
    cb0 = load_as<FT>(vb, s); cb1 = load_as<FT>(vb, s - si);
    fb = MY ? ba[s] : bb[s];
  }
  for (int k = k0; k < k1; k++, ss += sm) {
    u[5] = load_as<FT>(p.emf[PM], ss + 2 * sm);
    c[5] = load_as<FT>(p.emf[PM + 1], ss + 2 * sm);
    double iu[6], ic[6];
#pragma unroll
    for (int m = 0; m < 6; m++) {
      iu[m] = load_as<FT>(p.emf[PI], ss + (m - 3) * si);
      ic[m] = load_as<FT>(p.emf[PI + 1], ss + (m - 3) * si);
    }
    double ct = 0.5;
    if (ctw) {
      const double r0 = ro[ss], r1 = ro[ss - si];
      const double a0 = load_as<FT>(va, ss), a1 = load_as<FT>(va, ss - si);
      const double c0 = load_as<FT>(vb, ss), c1 = load_as<FT>(vb, ss - si);
      const double f0 = MY ? ba[ss] : bb[ss];        // the face B the marched axis steps over
      const double h0 = MY ? bb[ss] : ba[ss], h1 = MY ? bb[ss - si] : ba[ss - si];
      // cuct_weight's order: cells -xo-yo, -yo, -xo, 0; ba at -yo, 0; bb at -xo, 0
      if constexpr (MY) ct = cuct_weight(rb1, rb0, r1, r0, ab1, ab0, a1, a0, cb1, cb0, c1, c0, fb, f0, h1, h0);
      else ct = cuct_weight(rb1, r1, rb0, r0, ab1, a1, ab0, a0, cb1, c1, cb0, c0, h1, h0, fb, f0);
      rb0 = r0; rb1 = r1; ab0 = a0; ab1 = a1; cb0 = c0; cb1 = c1; fb = f0;
    }
    // Ez: x sweep B_y (t) along y, then y sweep B_x (u) along x;
    // Ey: x sweep B_z (u) along z, then z sweep B_x (t) along x;
    // Ex: y sweep B_z (t) along z, then z sweep B_y (u) along y:
    // a sweep's t part takes -1/2 and 1 - ct, its u part +1/2 and ct
    double ev = 0.0;
    ev += emf_part_w<ODR>(u, c, SM < 0 ? 1.0 - ct : ct, SM);
    ev += emf_part_w<ODR>(iu, ic, SI < 0 ? 1.0 - ct : ct, SI);
    store_as<FT>(E == 0 ? p.ex : (E == 1 ? p.ey : p.ez), ss, ev);
#pragma unroll
    for (int m = 0; m < 5; m++) {
      u[m] = u[m + 1];
      c[m] = c[m + 1];
    }
  }
}

// blocks: for each run of kc edges and each 256 edges of the plane, Ex, Ey and
// Ez in turn (Ez's runs are along y, its planes x-z)
template <int ODR, typename FT>
__global__ __launch_bounds__(256) void k_emf3d(StagePtrs p, Geo g, int ctw, int nbxy, int nbxz, int nxy, int kc)
{
  const int L = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  if (L < 2 * nxy) {
    const int b = L >> 1, chunk = b / nbxy;
    const unsigned q = (unsigned)(b - chunk * nbxy) * 256u + threadIdx.x;
    if (L & 1) emf3d_row<1, ODR, FT>(p, g, ctw, q, chunk, kc);
    else emf3d_row<0, ODR, FT>(p, g, ctw, q, chunk, kc);
  } else {
    const int b = L - 2 * nxy, chunk = b / nbxz;
    emf3d_row<2, ODR, FT>(p, g, ctw, (unsigned)(b - chunk * nbxz) * 256u + threadIdx.x, chunk, kc);
  }
}

// Large domains: all three components of the edges of a column in one thread,
// marching along z; the four z-interpolated face-part arrays sit in register
// windows and the cells of the plane behind are carried.  ro, v and B are read
// once for the three, where k_emf3d's Ez blocks, which run after the others,
// read them again; at 256 VGPRs (2 wavefronts per SIMD) and 32 planes a thread
// it needs many columns.  The line lies where a face-part array no longer stays
// in the caches: k_emf3d and this form take 279 and 292 us at 160^3 FP64 (38
// MB an array), 544 and 485 at 200^3 (72 MB), 8.92 and 6.47 ms at 512^3; mixed
// 338 and 348 us at 200^3 (36 MB), 368 and 361 at 64^2 x 2048 (43 MB), 507 and
// 472 at 224^3 (50 MB), 838 and 834 at 512^2 x 64 (78 MB), 5.43 and 4.51 ms at
// 512^3.  (In tiles of 64 x 4 columns, partly empty, it took 7.27 and 4.89 ms.)
constexpr long long EMF_ALL_MIN = 45000000;  // bytes of a face-part array
// Interpolate the face parts (upwind fu, central fc) of a
// sweep along axis o to the edge and combine with weight w:
//   sgn * ((uL + uR) + w (cL + cR))
template <int ODR, typename FT>
__device__ __forceinline__ double emf_part(const double* fu, const double* fc, long long ss, long long o, double w,
                                           double sgn)
{
  double a[5], b[5], ul0, ur0, ul1, ur1, dum;
#pragma unroll
  for (int m = 0; m < 5; m++) { a[m] = load_as<FT>(fu, ss + (m - 3) * o); b[m] = load_as<FT>(fc, ss + (m - 3) * o); }
  lin5<ODR>(a, ul0, dum);
  lin5<ODR>(b, ul1, dum);
#pragma unroll
  for (int m = 0; m < 5; m++) { a[m] = load_as<FT>(fu, ss + (m - 2) * o); b[m] = load_as<FT>(fc, ss + (m - 2) * o); }
  lin5<ODR>(a, dum, ur0);
  lin5<ODR>(b, dum, ur1);
  return sgn * ((ul0 + ur0) + w * (ul1 + ur1));
}

constexpr int EMF_KC = 32;  // planes per thread

template <int ODR, typename FT>
__global__ __launch_bounds__(256) void k_emf3d_z(StagePtrs p, Geo g, int ctw, int nbxy)
{
  const unsigned ni = (unsigned)g.nx - 5;  // edges on [3, n-3]
  const int L = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int chunk = L / nbxy;
  const unsigned q = (unsigned)(L - chunk * nbxy) * 256u + threadIdx.x;
  const unsigned row = q / ni;
  if (row >= (unsigned)g.ny - 5) return;  // no barriers below
  const int i = 3 + (int)(q - row * ni), j = 3 + (int)row;
  const int k0 = 3 + chunk * EMF_KC;
  const int k1 = k0 + EMF_KC < g.nz - 2 ? k0 + EMF_KC : g.nz - 2;
  const long long sy = g.sy, sz = g.sz;
  const double* ro = p.in[0];
  const double *bx = p.in[4], *by = p.in[5], *bz = p.in[6];
  // z windows at planes k-3 .. k+2
  double u2[6], c2[6], u4[6], c4[6];
  {
    const long long s0 = sz * k0 + sy * j + i;
#pragma unroll
    for (int m = 0; m < 5; m++) {
      const long long a = s0 + (m - 3) * sz;
      u2[m] = load_as<FT>(p.emf[2], a);
      c2[m] = load_as<FT>(p.emf[3], a);
      u4[m] = load_as<FT>(p.emf[4], a);
      c4[m] = load_as<FT>(p.emf[5], a);
    }
  }
  // plane k0-1 cell values used by the Ex / Ey weights
  double ro_p = 0, ro_pi = 0, ro_pj = 0, vx_p = 0, vx_pi = 0, vy_p = 0, vy_pj = 0, vz_p = 0, vz_pi = 0, vz_pj = 0,
         bx_p = 0, by_p = 0;
  if (ctw) {
    const long long s = sz * (k0 - 1) + sy * j + i;
    ro_p = ro[s]; ro_pi = ro[s - 1]; ro_pj = ro[s - sy];
    vx_p = load_as<FT>(p.vx, s); vx_pi = load_as<FT>(p.vx, s - 1);
    vy_p = load_as<FT>(p.vy, s); vy_pj = load_as<FT>(p.vy, s - sy);
    vz_p = load_as<FT>(p.vz, s); vz_pi = load_as<FT>(p.vz, s - 1); vz_pj = load_as<FT>(p.vz, s - sy);
    bx_p = bx[s]; by_p = by[s];
  }
  for (int k = k0; k < k1; k++) {
    const long long ss = sz * k + sy * j + i;
    {
      const long long a = ss + 2 * sz;
      u2[5] = load_as<FT>(p.emf[2], a);
      c2[5] = load_as<FT>(p.emf[3], a);
      u4[5] = load_as<FT>(p.emf[4], a);
      c4[5] = load_as<FT>(p.emf[5], a);
    }
    double ctz = 0.5, ctx = 0.5, cty = 0.5;
    double ro0 = 0, roi = 0, roj = 0, vx0 = 0, vxi = 0, vy0 = 0, vyj = 0, vz0 = 0, vzi = 0, vzj = 0, bx0 = 0,
           by0 = 0;
    if (ctw) {
      ro0 = ro[ss]; roi = ro[ss - 1]; roj = ro[ss - sy];
      const double roij = ro[ss - 1 - sy];
      vx0 = load_as<FT>(p.vx, ss); vxi = load_as<FT>(p.vx, ss - 1);
      const double vxj = load_as<FT>(p.vx, ss - sy), vxij = load_as<FT>(p.vx, ss - 1 - sy);
      vy0 = load_as<FT>(p.vy, ss); vyj = load_as<FT>(p.vy, ss - sy);
      const double vyi = load_as<FT>(p.vy, ss - 1), vyij = load_as<FT>(p.vy, ss - 1 - sy);
      vz0 = load_as<FT>(p.vz, ss); vzi = load_as<FT>(p.vz, ss - 1); vzj = load_as<FT>(p.vz, ss - sy);
      bx0 = bx[ss]; by0 = by[ss];
      // x-y plane for Ez: strides (1, ny)
      ctz = cuct_weight(roij, roj, roi, ro0, vxij, vxj, vxi, vx0, vyij, vyj, vyi, vy0, bx[ss - sy], bx0, by[ss - 1],
                        by0);
      // y-z plane for Ex: strides (sy, sz)
      ctx = cuct_weight(ro_pj, ro_p, roj, ro0, vy_pj, vy_p, vyj, vy0, vz_pj, vz_p, vzj, vz0, by_p, by0, bz[ss - sy],
                        bz[ss]);
      // z-x plane for Ey: strides (sz, 1)
      cty = cuct_weight(ro_pi, roi, ro_p, ro0, vz_pi, vzi, vz_p, vz0, vx_pi, vxi, vx_p, vx0, bz[ss - 1], bz[ss], bx_p,
                        bx0);
    }
    // Ez: x sweep B_y (t) along y, then y sweep B_x (u) along x
    double ez = 0.0;
    ez += emf_part<ODR, FT>(p.emf[0], p.emf[1], ss, sy, 1.0 - ctz, -0.5);
    ez += emf_part<ODR, FT>(p.emf[6], p.emf[7], ss, 1, ctz, +0.5);
    // Ey: x sweep B_z (u) along z, then z sweep B_x (t) along x
    double ey = 0.0;
    ey += emf_part_w<ODR>(u2, c2, cty, +0.5);
    ey += emf_part<ODR, FT>(p.emf[8], p.emf[9], ss, 1, 1.0 - cty, -0.5);
    // Ex: y sweep B_z (t) along z, then z sweep B_y (u) along y
    double ex = 0.0;
    ex += emf_part_w<ODR>(u4, c4, 1.0 - ctx, -0.5);
    ex += emf_part<ODR, FT>(p.emf[10], p.emf[11], ss, sy, ctx, +0.5);
    store_as<FT>(p.ex, ss, ex);
    store_as<FT>(p.ey, ss, ey);
    store_as<FT>(p.ez, ss, ez);
    // next plane: shift the windows, carry this plane's values
#pragma unroll
    for (int m = 0; m < 5; m++) {
      u2[m] = u2[m + 1];
      c2[m] = c2[m + 1];
      u4[m] = u4[m + 1];
      c4[m] = c4[m + 1];
    }
    ro_p = ro0; ro_pi = roi; ro_pj = roj;
    vx_p = vx0; vx_pi = vxi;
    vy_p = vy0; vy_pj = vyj;
    vz_p = vz0; vz_pi = vzi; vz_pj = vzj;
    bx_p = bx0; by_p = by0;
  }
}

// ------------------------------------------------------------------ CT
// Staggered-B update (mhd_updt3d_ctb, common/mhd_func.c:302-325), marching
// along z: one thread per (i, j) column of the x-y plane over kc planes.  The
// z-direction E values (Ey for bx, Ex for by) sit in 4-plane register windows,
// so each of those planes is read once per chunk instead of four times; the
// in-plane neighbours come through the caches.  Per face the operations and
// their order are those of the reference.
// FT: element type of the stored edge EMFs (the sweep precision)
template <int ODR, typename FT>
__global__ __launch_bounds__(256) void k_ct3d(StagePtrs p, Geo g, int nbxy, int kc)
{
  const unsigned ni = (unsigned)g.nx - 7;  // cells [4, n-4]
  const int L = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int chunk = L / nbxy;
  const unsigned q = (unsigned)(L - chunk * nbxy) * 256u + threadIdx.x;
  const unsigned row = q / ni;
  if (row >= (unsigned)g.ny - 7) return;  // no barriers below
  const int i = 4 + (int)(q - row * ni), j = 4 + (int)row;
  const int k0 = 4 + chunk * kc;
  const int k1 = k0 + kc < g.nz - 3 ? k0 + kc : g.nz - 3;
  const long long sy = g.sy, sz = g.sz;
  const long long c0 = sy * j + i;
  const double dtv = *p.dt;
  const double dtdx = dtv / g.dx, dtdy = dtv / g.dy, dtdz = dtv / g.dz;
  const FT *ex = reinterpret_cast<const FT*>(p.ex), *ey = reinterpret_cast<const FT*>(p.ey),
           *ez = reinterpret_cast<const FT*>(p.ez);
  const bool ji = j <= g.ny - 5, ii = i <= g.nx - 5;
  // windows: planes k-1 .. k+2 of ey and ex at (i, j); planes [3, nz-2]
  double eyw[4], exw[4];
#pragma unroll
  for (int m = 0; m < 3; m++) {
    eyw[m] = ey[c0 + sz * (k0 - 1 + m)];
    exw[m] = ex[c0 + sz * (k0 - 1 + m)];
  }
  for (int k = k0; k < k1; k++) {
    const long long ss = sz * k + c0;
    eyw[3] = ey[ss + 2 * sz];
    exw[3] = ex[ss + 2 * sz];
    const bool ki = k <= g.nz - 5;
    if (ji && ki) {  // bx: one extra face in x
      const double du0 = +dfc<ODR>((double)ez[ss - sy], (double)ez[ss], (double)ez[ss + sy], (double)ez[ss + 2 * sy]);
      const double du1 = -dfc<ODR>(eyw[0], eyw[1], eyw[2], eyw[3]);
      p.out[4][ss] = rk_upd(p.in[4][ss], p.u0[4][ss], -dtdy * du0 - dtdz * du1, p.a, p.b);
    }
    if (ii && ki) {  // by: one extra face in y
      const double du0 = +dfc<ODR>(exw[0], exw[1], exw[2], exw[3]);
      const double du1 = -dfc<ODR>((double)ez[ss - 1], (double)ez[ss], (double)ez[ss + 1], (double)ez[ss + 2]);
      p.out[5][ss] = rk_upd(p.in[5][ss], p.u0[5][ss], -dtdz * du0 - dtdx * du1, p.a, p.b);
    }
    if (ii && ji) {  // bz: one extra face in z
      const double du0 = +dfc<ODR>((double)ey[ss - 1], eyw[1], (double)ey[ss + 1], (double)ey[ss + 2]);
      const double du1 = -dfc<ODR>((double)ex[ss - sy], exw[1], (double)ex[ss + sy], (double)ex[ss + 2 * sy]);
      p.out[6][ss] = rk_upd(p.in[6][ss], p.u0[6][ss], -dtdx * du0 - dtdy * du1, p.a, p.b);
    }
#pragma unroll
    for (int m = 0; m < 3; m++) {
      eyw[m] = eyw[m + 1];
      exw[m] = exw[m + 1];
    }
  }
}

// ------------------------------------------------------------------ launch
typedef void (*sweep3_fn)(StagePtrs, Geo, BcFlags, double, int);

template <int DIR>
static sweep3_fn pick3(int rmn, int odr)
{
#define QAS_S(R, O) \
  if (rmn == R && odr == O) return DIR == 0 ? k_sweep3d<R, O, double> : k_sweep3d_t<DIR == 0 ? 1 : DIR, R, O, double>;
  QAS_S(0, 1) QAS_S(0, 2) QAS_S(0, 3) QAS_S(0, 4)
  QAS_S(1, 1) QAS_S(1, 2) QAS_S(1, 3) QAS_S(1, 4)
  QAS_S(2, 1) QAS_S(2, 2) QAS_S(2, 3) QAS_S(2, 4)
  QAS_S(3, 1) QAS_S(3, 2) QAS_S(3, 3) QAS_S(3, 4)
#undef QAS_S
  return nullptr;
}

static inline unsigned nblk3(long long n, int b) { return (unsigned)((n + b - 1) / b); }

// steps a marching thread takes: 32 amortise the filling of its windows, but
// few workgroups leave the chip waiting on each thread's chain of loads.  CT at
// 200^3 (mixed): 183 us with 1 428 workgroups, 174 with 2 054, 151 with 4 108,
// 143 with 8 058; at 128^3 97 with 495, 50 with 2 178 (4 steps).  The EMF (3
// components of more work each) gained nothing past 4 096.
static int march_chunk(long long plane_blocks, int n, int want)
{
  int kc = 32;
  while (kc > 4 && plane_blocks * ((n + kc - 1) / kc) < want) kc /= 2;
  return kc;
}

hipError_t launch_stage3d(qas_ctx* c, const StagePtrs& p)
{
  const Geo& g = c->geo;
  const int odr = c->s.odr;
  const double gam = c->s.gam;
  hipStream_t st = c->stream;
  const bool f32 = c->s.precision == 1;
  const int dims[3] = {g.nx, g.ny, g.nz};
  sweep3_fn f[3] = {pick3<0>(c->s.rmn, odr), pick3<1>(c->s.rmn, odr), pick3<2>(c->s.rmn, odr)};
  if (c->s.precision == 1)
    for (int d = 0; d < 3; d++) f[d] = pick_sweep_f32(3, d, c->s.rmn, odr);
  if (c->s.precision == 2)
    for (int d = 0; d < 3; d++) f[d] = pick_sweep_fma(3, d, c->s.rmn, odr);
  // z, then y, then x: the transverse sweeps leave dt/dz Dz and dt/dy Dy in
  // the accumulators, the x sweep applies the stage sum
  for (int d = 2; d >= 0; d--) {
    if (!f[d]) return hipErrorInvalidValue;
    if (d == 0) {
      QAS_LAUNCH(c, QAS_K_SWEEP_X, f[d], nblk3(g.nd, 256 - HALO), 256, x3_lds_bytes(f32), st, p, g, c->bc, gam, 0);
    } else {
      // one 256-thread workgroup per run of 60 cells of a 4-column group, in
      // every plane of the other transverse axis
      const int ncg = (g.nx + YC - 1) / YC, np = d == 1 ? g.nz : g.ny;
      const int bundle = line_bundle(ncg, dims[d], np);
      QAS_LAUNCH(c, QAS_K_SWEEP_X + d, f[d], (unsigned)(line_tiles(ncg, dims[d], bundle) * np), 256, 0, st, p, g, c->bc,
                 gam, bundle);
    }
  }
  // EMF and CT: 256 edges or cells of a plane per workgroup, march_chunk steps
  const int exy = (int)nblk3((long long)(g.nx - 5) * (g.ny - 5), 256), exz = (int)nblk3((long long)(g.nx - 5) * (g.nz - 5), 256);
  const int ek = march_chunk(3LL * exy, g.nz - 5, 4096);
  const int nexy = exy * (int)nblk3(g.nz - 5, ek);
  const unsigned nemf = (unsigned)(2 * nexy + exz * (int)nblk3(g.ny - 5, ek));
  const int cxy = (int)nblk3((long long)(g.nx - 7) * (g.ny - 7), 256);
  const int ck = march_chunk(cxy, g.nz - 7, 8192);
  const unsigned nct = (unsigned)(cxy * (int)nblk3(g.nz - 7, ck));
  const unsigned nemfz = (unsigned)(exy * (int)nblk3(g.nz - 5, EMF_KC));
  const bool all = g.nd * (f32 ? 4 : 8) >= EMF_ALL_MIN;
  // (the face parts and edges are stored in the sweep precision)
#define QAS_EMF_CT(O)                                                                                             \
  if (all && f32) QAS_LAUNCH(c, QAS_K_EMF, (k_emf3d_z<O, float>), nemfz, 256, 0, st, p, g, c->s.ctw, exy);             \
  else if (all) QAS_LAUNCH(c, QAS_K_EMF, (k_emf3d_z<O, double>), nemfz, 256, 0, st, p, g, c->s.ctw, exy);              \
  else if (f32) QAS_LAUNCH(c, QAS_K_EMF, (k_emf3d<O, float>), nemf, 256, 0, st, p, g, c->s.ctw, exy, exz, nexy, ek);   \
  else QAS_LAUNCH(c, QAS_K_EMF, (k_emf3d<O, double>), nemf, 256, 0, st, p, g, c->s.ctw, exy, exz, nexy, ek);      \
  if (f32) QAS_LAUNCH(c, QAS_K_CT, (k_ct3d<O, float>), nct, 256, 0, st, p, g, cxy, ck);                           \
  else QAS_LAUNCH(c, QAS_K_CT, (k_ct3d<O, double>), nct, 256, 0, st, p, g, cxy, ck);
  switch (odr) {
    case 1: QAS_EMF_CT(1) break;
    case 2: QAS_EMF_CT(2) break;
    case 3: QAS_EMF_CT(3) break;
    default: QAS_EMF_CT(4) break;
  }
#undef QAS_EMF_CT
  return hipGetLastError();
}

}  // namespace qas
