// qas_sweep3d.hpp -- the 3D face sweep kernel, templated on the precision T
// of the reconstruction and Riemann solver (double: FP64 path; float: mixed
// path).  Included by qas_kernels3d.hip and qas_mixed.hip.
#pragma once
#include "qas_device.hpp"
#include "qas_internal.hpp"
#include "qas_sweep2d.hpp"

namespace qas {

// dv of axis A (0 x, 1 y, 2 z) at (i, j, k) after its bound()
// (mhd3d_solve.cpp:138-164): flags (-dnxs[1], dnys[1], dnzs[1]) for dvx,
// (dnxs[2], -dnys[2], dnzs[2]) for dvy, (dnxs[3], dnys[3], -dnzs[3]) for dvz.
// v: the velocity array, or a VelOf reading it from the state.
template <int A, typename V>
__device__ __forceinline__ double dv3(const V& v, int i, int j, int k, const Geo& g, const BcFlags& bc)
{
  using VT = typename std::remove_cv<typename std::remove_reference<decltype(v[0])>::type>::type;
  const int dnx = A == 0 ? -bc.dn[0][1] : bc.dn[0][1 + A];
  const int dny = A == 1 ? -bc.dn[1][2] : bc.dn[1][1 + A];
  const int dnz = A == 2 ? -bc.dn[2][3] : bc.dn[2][1 + A];
  const Src sx = resolve(i, g.nx, 0, dnx);
  const Src sy = resolve(j, g.ny, 0, dny);
  const Src sz = resolve(k, g.nz, 0, dnz);
  const long long q = g.sz * sz.i + g.sy * sy.i + sx.i;
  const long long o = A == 0 ? 1 : (A == 1 ? g.sy : g.sz);
  const VT r = tmin((VT)(v[q + o] - v[q]), (VT)(v[q] - v[q - o]));
  return apply(sz, apply(sy, apply(sx, (double)r)));
}

// the same from the state (velocity m (1/ro) rounded to VT, the stored
// primitive's value), for the sweep that stores the primitives
template <int A, typename VT>
__device__ __forceinline__ double dv3_state(const StagePtrs& p, int i, int j, int k, const Geo& g, const BcFlags& bc)
{
  return dv3<A>(VelOf<VT>{p.in[1 + A], p.in[0]}, i, j, k, g, bc);
}

// the sensor of cell (i, j, k) for the faces along DIR: the smaller of the
// two transverse axes' dv (STATE: velocities from the state)
template <int DIR, bool STATE, typename VT>
__device__ __forceinline__ VT dv3_cell(const StagePtrs& p, int i, int j, int k, const Geo& g, const BcFlags& bc)
{
  constexpr int TA = (DIR + 1) % 3, TB = (DIR + 2) % 3;
  const PrimView<VT> pv = prim_view<VT>(p);
  const VT* vax[3] = {pv.vx, pv.vy, pv.vz};
  double a, b;
  if constexpr (STATE) {
    a = dv3_state<TA, VT>(p, i, j, k, g, bc);
    b = dv3_state<TB, VT>(p, i, j, k, g, bc);
  } else {
    a = dv3<TA>(vax[TA], i, j, k, g, bc);
    b = dv3<TB>(vax[TB], i, j, k, g, bc);
  }
  return (VT)tmin(a, b);
}

// Cell-centred B (fcen along x, y, z on the staggered components, then the
// bound() index map at ghost cells) and primitives of cell (i, j, k) = flat
// index t from the stage input state (mhd_class.hpp:80-91, mhd_func.c:6-16;
// mhd3d_solve.cpp:49-98), FP64 with the reference's operation order in every
// precision (no FMA contraction here).  INNER: the caller knows the cell is
// no ghost cell, where the index map is the identity.
struct Prim3d {
  double vx, vy, vz, pr, c[3];
};

template <int ODR, bool INNER>
__device__ __forceinline__ Prim3d prim3d_cell(const StagePtrs& p, const Geo& g, const BcFlags& bc, double gam, int i,
                                              int j, int k, long long t)
{
#pragma clang fp contract(off)
  Prim3d r;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const double* b = p.in[4 + a];
    const long long o = a == 0 ? 1 : (a == 1 ? g.sy : g.sz);
    if constexpr (INNER) {
      r.c[a] = fcen<ODR>(b[t - o], b[t], b[t + o], b[t + 2 * o]);
    } else {
      const Src sx = resolve(i, g.nx, 0, bc.dn[0][4 + a]);
      const Src sy = resolve(j, g.ny, 0, bc.dn[1][4 + a]);
      const Src sz = resolve(k, g.nz, 0, bc.dn[2][4 + a]);
      const long long q = g.sz * sz.i + g.sy * sy.i + sx.i;
      const double v = fcen<ODR>(b[q - o], b[q], b[q + o], b[q + 2 * o]);
      r.c[a] = apply(sz, apply(sy, apply(sx, v)));
    }
  }
  const double ro = p.in[0][t];
  const double iro = FastOps::inv(ro);
  r.vx = p.in[1][t] * iro;
  r.vy = p.in[2][t] * iro;
  r.vz = p.in[3][t] * iro;
  const double v2 = r.vx * r.vx + r.vy * r.vy + r.vz * r.vz;
  const double b2 = r.c[0] * r.c[0] + r.c[1] * r.c[1] + r.c[2] * r.c[2];
  r.pr = (gam - 1) * (p.in[7][t] - 0.5 * (ro * v2 + b2));
  return r;
}

// ------------------------------------------------------------------ y, z sweeps
// LDS-staged as the 2D y sweep (qas_sweep2d.hpp): one workgroup = 4
// wavefronts = 4 adjacent x-columns x one run of 60 cells along DIR
// (line_tile, in the plane of x and DIR) at one position of the other
// transverse axis; stencil inputs loaded cooperatively (4 consecutive values
// of a row per 4 threads) into LDS, fluxes and face parts staged in LDS,
// differenced and written back by coalesced threads.  Bit-identical to a
// direct per-lane sweep.  z and y sweeps at 128^3 (FP64) 302 and 228 us with
// runs cut by column and shuffles, 257 and 196 this way; at 200^3 (mixed, the
// tile in FP32) 602 and 447 -> 562 and 329.
// Column length of the results in LDS: 64 are used; 70, with the tile's 72, lets
// four FP64 workgroups into a CU's 160 KB (at 72 three: 128^3 HLLD ODR 1 y 139.6 us
// against 129.9, ODR 3 184 against 170; at 64 the write-back's 4 columns fall
// on the same banks, Roe 1 to 2 % slower).
constexpr int YO3 = 70;
template <int DIR, int RMN, int ODR, typename T>
__device__ __forceinline__ void sweep3d_t(const StagePtrs& p, const Geo& g, const BcFlags& bc, double gam, int bundle)
{
  static_assert(DIR == 1 || DIR == 2, "transverse sweeps only");
  constexpr int TA = (DIR + 1) % 3;
  constexpr int TB = (DIR + 2) % 3;
  constexpr int LB = DIR == 2 ? 1 : 2;  // the other transverse axis (x is the column axis)
  __shared__ T sh[9][YC][YRP];      // ro vn vt vu bt bu pr cn bf
  __shared__ T so[9][YC][YO3];      // 5 fluxes, 4 face parts
  const int dims[3] = {g.nx, g.ny, g.nz};
  const long long strd[3] = {1, g.sy, g.sz};
  const int ncg = (g.nx + YC - 1) / YC;
  const int nlb = dims[LB], n = dims[DIR];
  const int L = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int nt = line_tiles(ncg, n, bundle);
  if (L >= nt * nlb) return;  // whole workgroup
  const int lb = L / nt;
  const LineTile tl = line_tile(L - lb * nt, ncg, n, bundle);
  const long long o = strd[DIR];
  const long long blb = strd[LB] * lb;
  const PrimView<T> pv = prim_view<T>(p);
  const T* vax[3] = {pv.vx, pv.vy, pv.vz};
  const T* cax[3] = {pv.cx, pv.cy, pv.cz};
  if constexpr (DIR == 2) {
    // The z sweep runs first: its staging computes the primitives of the
    // tile's cells from the stage input state and rounds them once to T; the
    // run's own cells (its x-columns at this y) are stored for the y and x
    // sweeps, so every cell is written once.
    const bool inner = (tl.col * YC >= NG) && (tl.col * YC + YC - 1 <= g.nx - NG - 1) && (tl.row - 4 >= NG) &&
                       (tl.row + YR - 5 <= n - NG - 1) && (lb >= NG) && (lb <= nlb - NG - 1);
    for (int e = threadIdx.x; e < YC * YR; e += blockDim.x) {
      const int c = e % YC, r = e / YC;
      int cg, row;
      line_cell(tl, n, r - 4, cg, row);
      const int colu = cg * YC + c;
      const int col = colu > g.nx - 1 ? g.nx - 1 : colu;
      const long long a = blb + o * row + col;
      const Prim3d q = inner ? prim3d_cell<ODR, true>(p, g, bc, gam, col, lb, row, a)
                             : prim3d_cell<ODR, false>(p, g, bc, gam, col, lb, row, a);
      const T v3[3] = {(T)q.vx, (T)q.vy, (T)q.vz};
      const T c3[3] = {(T)q.c[0], (T)q.c[1], (T)q.c[2]};
      const T pr = (T)q.pr;
      sh[0][c][r] = (T)p.in[0][a];
      sh[1][c][r] = v3[DIR];
      sh[2][c][r] = v3[TA];
      sh[3][c][r] = v3[TB];
      sh[4][c][r] = c3[TA];
      sh[5][c][r] = c3[TB];
      sh[6][c][r] = pr;
      sh[7][c][r] = c3[DIR];
      sh[8][c][r] = (T)p.in[4 + DIR][a];
      if (colu < g.nx && r - 4 >= tl.lo && r - 4 < tl.hi) {
        reinterpret_cast<T*>(p.vx)[a] = v3[0];
        reinterpret_cast<T*>(p.vy)[a] = v3[1];
        reinterpret_cast<T*>(p.vz)[a] = v3[2];
        reinterpret_cast<T*>(p.pr)[a] = pr;
        reinterpret_cast<T*>(p.cx)[a] = c3[0];
        reinterpret_cast<T*>(p.cy)[a] = c3[1];
        reinterpret_cast<T*>(p.cz)[a] = c3[2];
      }
    }
  } else {
    const T* src[6] = {vax[DIR], vax[TA], vax[TB], cax[TA], cax[TB], pv.pr};
    for (int e = threadIdx.x; e < YC * YR; e += blockDim.x) {
      const int c = e % YC, r = e / YC;
      int cg, row;
      line_cell(tl, n, r - 4, cg, row);
      int col = cg * YC + c;
      col = col > g.nx - 1 ? g.nx - 1 : col;
      const long long a = blb + o * row + col;
      sh[0][c][r] = (T)p.in[0][a];
#pragma unroll
      for (int k = 0; k < 6; k++) sh[1 + k][c][r] = src[k][a];
      sh[7][c][r] = cax[DIR][a];
      sh[8][c][r] = (T)p.in[4 + DIR][a];
    }
  }
  __syncthreads();
  const int w = threadIdx.x / WAVE;
  const int lane = threadIdx.x & (WAVE - 1);
  const int rb = lane + 2;  // this lane's cell in the tile
  // FP32 reads its stencil from LDS field by field, FP64 holds it in registers
  constexpr bool IN_LDS = sizeof(T) == 4;
  const LdsStencil<T, T, YC * YRP, 1> sl{&sh[0][w][rb]};
  T sr[7][5];
  if constexpr (!IN_LDS) {
#pragma unroll
    for (int m = 0; m < 5; m++)
#pragma unroll
      for (int k = 0; k < 7; k++) sr[k][m] = sl(k, m);
  }
  const auto s = [&]() {
    if constexpr (IN_LDS) return sl;
    else return RegStencil<T>{sr};
  }();
  // B-flux face states for both tangential components (mhd_lr_fb)
  T qlt, qrt, qlu, qru;
  {
    const T bnm = sh[8][w][rb], bnp = sh[8][w][rb + 1];
    T pp[5], qq[5];
#pragma unroll
    for (int m = 0; m < 5; m++) {
      pp[m] = s(4, m) * s(1, m);
      qq[m] = s(2, m);
    }
    lr_fb<ODR>(pp, qq, bnm, bnp, qlt, qrt);
#pragma unroll
    for (int m = 0; m < 5; m++) {
      pp[m] = s(5, m) * s(1, m);
      qq[m] = s(3, m);
    }
    lr_fb<ODR>(pp, qq, bnm, bnp, qlu, qru);
  }
  // central parts of the face's B fluxes
  const T fct = T(0.5) * ((T)__shfl_up(qlt, 1, WAVE) + qrt);
  const T fcu = T(0.5) * ((T)__shfl_up(qlu, 1, WAVE) + qru);
  so[6][w][lane] = fct;
  so[8][w][lane] = fcu;
  s.again();
  T vl[7], vr[7];
  lrstate_of<ODR, T, 0, true, std::is_same<T, double>::value>(s, sh[7][w][rb], (T)gam, vl, vr);
  T Lf[7], F[7];
#pragma unroll
  for (int k = 0; k < 7; k++) Lf[k] = __shfl_up(vl[k], 1, WAVE);
  const T bnf = sh[8][w][rb];  // (both sides of the face share it)
  T dv0 = T(0.0), dv1 = T(0.0);
  if constexpr (RMN >= 2) {
    dv0 = sh[1][w][rb] - sh[1][w][rb - 1];
    // the sensor of this lane's cell; the other one of its face is the lane
    // before's.  (z sweep: the velocities of the neighbouring columns are
    // being stored by other workgroups of this launch: from the state)
    int cg, q;
    line_cell(tl, n, lane - 2, cg, q);
    int c0[3];
    c0[0] = cg * YC + w > g.nx - 1 ? g.nx - 1 : cg * YC + w;
    c0[LB] = lb;
    c0[DIR] = q;
    const T dvc = dv3_cell<DIR, DIR == 2, T>(p, c0[0], c0[1], c0[2], g, bc);
    dv1 = tmin((T)__shfl_up(dvc, 1, WAVE), dvc);
  }
  riemann<RMN>(Lf, vr, bnf, (T)gam, dv0, dv1, F);
  so[5][w][lane] = F[4] - fct;
  so[7][w][lane] = F[5] - fcu;
  so[0][w][lane] = F[0];
  so[1 + DIR][w][lane] = F[1];
  so[1 + TA][w][lane] = F[2];
  so[1 + TB][w][lane] = F[3];
  so[4][w][lane] = F[6];
  __syncthreads();
  {
    const int c = threadIdx.x % YC, r = threadIdx.x / YC;
    int cg, row;
    line_cell(tl, n, r - 2, cg, row);
    const int i = cg * YC + c;
    const bool own = (r >= 2) && (r - 2 < tl.hi) && (r < 2 + SEG) && (row >= 3) && (row <= n - 3) && (i < g.nx);
    if (own) {
      const long long a = blb + o * row + i;
#pragma unroll
      for (int k = 0; k < 4; k++) store_as<T>(p.emf[DIR * 4 + k], a, so[5 + k][c][r]);
      const bool upd = (row >= NG) && (row <= n - NG - 1) && (i >= NG) && (i <= g.nx - NG - 1) && (lb >= NG) &&
                       (lb <= nlb - NG - 1);
      if (upd) {
        // dt/dy Dy (slots 0-4) or dt/dz Dz (slots 5-9) of (ro, mx, my, mz,
        // en); the x sweep, which runs last, subtracts both
        const double dtd = *p.dt / (DIR == 1 ? g.dy : g.dz);
        double* const* acc = p.acc + (DIR == 1 ? 0 : 5);
#pragma unroll
        for (int v = 0; v < 5; v++)
          store_as<T>(acc[v], a, dtd * dfc<ODR>((double)so[v][c][r - 1], (double)so[v][c][r], (double)so[v][c][r + 1],
                                                (double)so[v][c][r + 2]));
      }
    }
  }
}

// FMA: build tag of the instantiation (see k_sweep2d_y)
template <int DIR, int RMN, int ODR, typename T, int FMA = 0>
__global__ __launch_bounds__(256, 2) void k_sweep3d_t(StagePtrs p, Geo g, BcFlags bc, double gam, int bundle)
{
  sweep3d_t<DIR, RMN, ODR, T>(p, g, bc, gam, bundle);
}

// ------------------------------------------------------------------ x sweep
// Runs of the domain's cells in memory order, states and fluxes handed over
// through LDS as in the 2D x sweep; it runs after the z and y sweeps and
// applies the RK stage sum.  128^3 (FP64) 272 -> 186 us, 200^3 (mixed) 448 -> 386.
// Waves per SIMD: FP32 MLAU below ODR 4 needs 5 (128^3, ODR 3 113 us against 126;
// ODR 4 takes 121 VGPRs).
template <int RMN, int ODR, typename T, int FMA = 0>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? (RMN == 3 && ODR < 4 ? 5 : 4) : (RMN == 1 ? 3 : 2)) void k_sweep3d(StagePtrs p, Geo g, BcFlags bc, double gam, int)
{
  extern __shared__ double x_lds[];
  constexpr int XL3 = 11;  // 7 states, 2 B-flux states, the sensor; odd
  const int nb = (int)blockDim.x;
  T* const xs = reinterpret_cast<T*>(x_lds) + XS * ((int)threadIdx.x + 2);                // this lane's cell
  T* const xl = reinterpret_cast<T*>(x_lds) + XS * (nb + HALO) + XL3 * (int)threadIdx.x;  // its face values
  const int n = g.nx;
  const XCell cell = x_cell((int)blockIdx.x, n, g.nd);
  const int q = cell.i;
  const int k = (int)((unsigned)cell.row / (unsigned)g.ny), j = cell.row - k * g.ny;
  const long long base = cell.a - q;  // the row's first cell

  const PrimView<T> pv = prim_view<T>(p);
  const double* bf = p.in[4];
  auto load = [&](int v, long long a) -> T {
    switch (v) {
      case 0: return (T)p.in[0][a];
      case 1: return pv.vx[a];
      case 2: return pv.vy[a];
      case 3: return pv.vz[a];
      case 4: return pv.cy[a];
      case 5: return pv.cz[a];
      default: return pv.pr[a];
    }
  };
  T sr[7][5];
  if constexpr (sizeof(T) == 8) {
    const long long sc = base + (q < 2 ? 2 : (q > n - 3 ? n - 3 : q));
#pragma unroll
    for (int m = 0; m < 5; m++)
#pragma unroll
      for (int v = 0; v < 7; v++) sr[v][m] = load(v, sc + (m - 2));
  } else {
#pragma unroll
    for (int v = 0; v < 7; v++) xs[v] = load(v, cell.a);
    if (threadIdx.x < HALO) {  // the 2 cells before the first lane's and the 2 after the last one's
      const int d = threadIdx.x < 2 ? (int)threadIdx.x - 2 : nb + (int)threadIdx.x - 2;
      long long a = (long long)blockIdx.x * (nb - HALO) - 2 + d;
      a = a < 0 ? 0 : (a > g.nd - 1 ? g.nd - 1 : a);
#pragma unroll
      for (int v = 0; v < 7; v++) reinterpret_cast<T*>(x_lds)[XS * (d + 2) + v] = load(v, a);
    }
  }
  const T cn = pv.cx[cell.a], bm = (T)bf[cell.a], bp = (T)bf[cell.a + 1 < g.nd ? cell.a + 1 : cell.a];
  if constexpr (sizeof(T) == 4) __syncthreads();
  const auto s = [&]() {
    if constexpr (sizeof(T) == 8) return RegStencil<T>{sr};
    else return LdsStencil<T, T, 1, XS>{xs};
  }();
  // B-flux face states for both tangential components (mhd_lr_fb)
  T qrt, qru;
  {
    T pp[5], qq[5], ql;
#pragma unroll
    for (int m = 0; m < 5; m++) {
      pp[m] = s(4, m) * s(1, m);
      qq[m] = s(2, m);
    }
    lr_fb<ODR>(pp, qq, bm, bp, ql, qrt);
    xl[7] = ql;
#pragma unroll
    for (int m = 0; m < 5; m++) {
      pp[m] = s(5, m) * s(1, m);
      qq[m] = s(3, m);
    }
    lr_fb<ODR>(pp, qq, bm, bp, ql, qru);
    xl[8] = ql;
  }
  const T vnf = s(1, 2), vnb = s(1, 1);  // of the face's two cells
  T dvc = T(0.0);  // the transverse sensor of this lane's cell
  if constexpr (RMN >= 2) {
    dvc = dv3_cell<0, false, T>(p, q, j, k, g, bc);
    xl[9] = dvc;
  }
  s.again();
  T vl[7], vr[7];
  lrstate_of<ODR, T, 0, true, std::is_same<T, double>::value>(s, cn, (T)gam, vl, vr);
#pragma unroll
  for (int v = 0; v < 7; v++) xl[v] = vl[v];
  __syncthreads();
  const T* const xb = threadIdx.x > 0 ? xl - XL3 : xl;  // (lane 0's flux is not used)
  T L[7], F[7];
#pragma unroll
  for (int v = 0; v < 7; v++) L[v] = xb[v];
  const T fct = T(0.5) * (xb[7] + qrt);
  const T fcu = T(0.5) * (xb[8] + qru);
  T dv0 = T(0.0), dv1 = T(0.0);
  if constexpr (RMN >= 2) {
    dv0 = vnf - vnb;
    dv1 = tmin(xb[9], dvc);
  }
  riemann<RMN>(L, vr, bm, (T)gam, dv0, dv1, F);
  const bool own = cell.own && (q >= 3) && (q <= n - 3);
  if (own) {
    store_as<T>(p.emf[0], cell.a, (double)(F[4] - fct));  // B_t flux, upwind part
    store_as<T>(p.emf[1], cell.a, (double)fct);           // B_t flux, central part
    store_as<T>(p.emf[2], cell.a, (double)(F[5] - fcu));  // B_u flux, upwind part
    store_as<T>(p.emf[3], cell.a, (double)fcu);           // B_u flux, central part
  }
  // divergence of ro, mx, my, mz, en (every lane has read its stencil)
  const int fid[5] = {0, 1, 2, 3, 6};
#pragma unroll
  for (int v = 0; v < 5; v++) xs[v] = F[fid[v]];
  __syncthreads();
  const bool upd = own && (q >= NG) && (q <= n - NG - 1) && (j >= NG) && (j <= g.ny - NG - 1) && (k >= NG) &&
                   (k <= g.nz - NG - 1);
  if (!upd) return;
  // the z and y sweeps ran first (dt/dz Dz in slots 5-9, dt/dy Dy in 0-4);
  // the stage sum u = a u0 + b (u + (((-dt/dx Dx) - dt/dy Dy) - dt/dz Dz))
  // is the reference's expression in its order (mhd3d_solve.cpp:658-676)
  const long long c = cell.a;
  const double dtdx = *p.dt / g.dx;
  const int vid[5] = {0, 1, 2, 3, 7};
#pragma unroll
  for (int v = 0; v < 5; v++) {
    const int m = vid[v];
    const double du = dfc<ODR>((double)xs[v - XS], (double)F[fid[v]], (double)xs[v + XS], (double)xs[v + 2 * XS]);
    p.out[m][c] = rk_upd(p.in[m][c], p.u0[m][c], ((-dtdx * du) - load_as<T>(p.acc[v], c)) - load_as<T>(p.acc[5 + v], c),
                         p.a, p.b);
  }
}

constexpr unsigned x3_lds_bytes(bool f32) { return (unsigned)((XS * (256 + HALO) + 11 * 256) * (f32 ? 4 : 8)); }

}  // namespace qas
