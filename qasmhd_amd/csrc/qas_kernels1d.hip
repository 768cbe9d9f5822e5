// qas_kernels1d.hip -- one SSP-RK stage of the 1D ideal-MHD step on gfx950.
//
// Replaces the stage body of MHD1D::ideal (1D/SERIAL/shock/mhd1d_solve.cpp:
// 99-184) in one launch: primitives (:104-112), reconstruction of each cell
// (:113-141), the flux of each face (:142-162), the 4th-order difference and
// RK stage sum of the seven evolved variables (:163-179) and the ghost fill of
// the stage output (:181-183).  In 1D the cell-centred B is the stored B
// (cx=bx, cy=by, cz=bz, :89-91) and bx is not evolved (it is carried into the
// stage output buffer).
#include "qas_device.hpp"
#include "qas_internal.hpp"
#include "qas_stage2d.hpp"

namespace qas {

// One workgroup of one wavefront per 60 cells.  A domain of some thousand cells is a handful of
// wavefronts, so a step is latency: as three launches a stage (primitives 2.6
// us, sweep 9.6, ghost fill 4.0, and the gaps) 32 steps of 1024 cells took 1.76
// ms, as one launch (12.0 us) 1.40.  The wavefront stages its 68 cells' primitives in LDS (each lane
// its own and one more, so that both sets of loads are in flight together), and
// a lane whose cell bound() copies writes the ghosts itself.
template <int RMN, int ODR>
__global__ __launch_bounds__(WAVE) void k_stage1d(StagePtrs p, Geo g, BcFlags bc, double gam)
{
  __shared__ double sh[7][WAVE + HALO];  // ro vx vy vz by bz pr
  const int lane = threadIdx.x, seg = (int)blockIdx.x;
  const int n = g.nx;
  const int f0 = 3 + seg * SEG;
  const int q = f0 - 2 + lane;  // this lane's cell
  {
    const int r1 = lane < HALO ? WAVE + lane : lane;  // the last 4 places are lanes 0..3's
    const int place[2] = {lane, r1};
    double u[2][8];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int c = f0 - 4 + place[e];
      const int a = c < 0 ? 0 : (c > n - 1 ? n - 1 : c);
#pragma unroll
      for (int m = 0; m < 8; m++) u[e][m] = p.in[m][a];
    }
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const double iro = FastOps::inv(u[e][0]);
      const double vx = u[e][1] * iro, vy = u[e][2] * iro, vz = u[e][3] * iro;
      const double v2 = vx * vx + vy * vy + vz * vz;
      const double b2 = u[e][4] * u[e][4] + u[e][5] * u[e][5] + u[e][6] * u[e][6];
      double* const to = &sh[0][place[e]];
      constexpr int R = WAVE + HALO;
      to[0] = u[e][0];
      to[R] = vx;
      to[2 * R] = vy;
      to[3 * R] = vz;
      to[4 * R] = u[e][5];
      to[5 * R] = u[e][6];
      to[6 * R] = (gam - 1) * (u[e][7] - 0.5 * (u[e][0] * v2 + b2));
    }
  }
  __syncthreads();
  const double* bx = p.in[4];
  const int qc = q < 0 ? 0 : (q > n - 1 ? n - 1 : q);
  const double bn = bx[qc];
  double s[7][5];
#pragma unroll
  for (int m = 0; m < 5; m++)
#pragma unroll
    for (int k = 0; k < 7; k++) s[k][m] = sh[k][lane + m];
  double vl[7], vr[7];
  lrstate<ODR>(s, bn, gam, vl, vr);
  double L[7], F[7];
#pragma unroll
  for (int k = 0; k < 7; k++) L[k] = __shfl_up(vl[k], 1, WAVE);
  const double dv0 = s[1][2] - s[1][1];
  riemann<RMN>(L, vr, bn, gam, dv0, 0.0, F);
  // evolved: ro, mx, my, mz, by, bz, en = F0..F6
  double du[7];
#pragma unroll
  for (int v = 0; v < 7; v++) {
    const double fm1 = __shfl_up(F[v], 1, WAVE);
    const double f1 = __shfl_down(F[v], 1, WAVE);
    const double f2 = __shfl_down(F[v], 2, WAVE);
    du[v] = dfc<ODR>(fm1, F[v], f1, f2);
  }
  const bool own = (lane >= 2) && (lane < 2 + SEG) && (q >= NG) && (q <= n - NG);
  if (!own) return;
  const bool upd = q <= n - NG - 1;  // cell n - 4 is at most kept (a staggered variable's last face)
  const double dtdx = *p.dt / g.dx;
  constexpr int flux_of[8] = {0, 1, 2, 3, -1, 4, 5, 6};
#pragma unroll
  for (int m = 0; m < 8; m++) {
    const int st = bc.st[0][m], dn = bc.dn[0][m];
    if (!upd && resolve(q, n, st, dn).i != q) continue;  // a ghost of this variable
    double v;
    if (m == 4) v = bn;
    else if (upd) v = rk_upd(p.in[m][q], p.u0[m][q], -dtdx * du[flux_of[m] < 0 ? 0 : flux_of[m]], p.a, p.b);
    else v = p.out[m][q];
    p.out[m][q] = v;
    // the ghosts that bound() copies from this cell
    if (q < 2 * NG + 1 || q >= n - 2 * NG - 1) {
      const Src f = resolve(0, n, st, dn);  // its factor, the same at both ends
      for (unsigned x = ghost_images(q, n, st, dn); x; x &= x - 1) {
        const int a = __builtin_ctz(x);
        p.out[m][a < NG ? a : n - 2 * NG + a] = apply(f, v);
      }
    }
  }
}

typedef void (*sweep1_fn)(StagePtrs, Geo, BcFlags, double);

static sweep1_fn pick1(int rmn, int odr)
{
#define QAS_S(R, O) \
  if (rmn == R && odr == O) return k_stage1d<R, O>;
  QAS_S(0, 1) QAS_S(0, 2) QAS_S(0, 3) QAS_S(0, 4)
  QAS_S(1, 1) QAS_S(1, 2) QAS_S(1, 3) QAS_S(1, 4)
  QAS_S(2, 1) QAS_S(2, 2) QAS_S(2, 3) QAS_S(2, 4)
  QAS_S(3, 1) QAS_S(3, 2) QAS_S(3, 3) QAS_S(3, 4)
#undef QAS_S
  return nullptr;
}

hipError_t launch_stage1d(qas_ctx* c, const StagePtrs& p)
{
  const Geo& g = c->geo;
  const int nseg = (g.nx - 5 + SEG - 1) / SEG;
  sweep1_fn f = pick1(c->s.rmn, c->s.odr);
  if (!f) return hipErrorInvalidValue;
  QAS_LAUNCH(c, QAS_K_SWEEP_X, f, (unsigned)nseg, WAVE, 0, c->stream, p, g, c->bc, c->s.gam);
  return hipGetLastError();
}

}  // namespace qas
