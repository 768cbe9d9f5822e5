// qas_sweep2d.hpp -- the 2D face sweep kernel, templated on the precision T
// of the reconstruction and Riemann solver (double: the FP64 path, bit-
// identical to the reference; float: the mixed path).  Included by
// qas_kernels2d.hip (T = double, -ffp-contract=off) and qas_mixed.hip
// (T = float).  A lane reconstructs one cell, takes the left state of its face
// from the lane before and the four fluxes of its difference from its
// neighbours, so the 2 outer lanes on each side of a run of cells only feed
// the others: a run is one wavefront along y and a whole workgroup along x.
#pragma once
#include "qas_batch.hpp"
#include "qas_device.hpp"
#include "qas_internal.hpp"
#include "qas_stage2d.hpp"

namespace qas {

// velocity component m (1/ro) of a cell from the state, rounded to T as
// the stored primitive is
template <typename T>
struct VelOf {
  const double* m;
  const double* ro;
  __device__ __forceinline__ T operator[](long long q) const { return (T)(m[q] * FastOps::inv(ro[q])); }
};

// shock sensor dv of mhd2d_solve.cpp:105-125 at (i, j) after its bound():
// DIR 0 -> dvx (flags -dnxs[1], dnys[1]); DIR 1 -> dvy (dnxs[2], -dnys[2]).
// v: the velocity array, or a VelOf<VT> reading it from the state.
template <int DIR, typename V>
__device__ __forceinline__ double dv_at(const V& v, int i, int j, const Geo& g, const BcFlags& bc)
{
  using VT = typename std::remove_cv<typename std::remove_reference<decltype(v[0])>::type>::type;
  const int dnx = DIR == 0 ? -bc.dn[0][1] : bc.dn[0][2];
  const int dny = DIR == 0 ? bc.dn[1][1] : -bc.dn[1][2];
  const Src sx = resolve(i, g.nx, 0, dnx);
  const Src sy = resolve(j, g.ny, 0, dny);
  const long long q = (long long)g.nx * sy.i + sx.i;
  const long long o = DIR == 0 ? 1 : g.nx;
  const VT r = tmin((VT)(v[q + o] - v[q]), (VT)(v[q] - v[q - o]));
  return apply(sy, apply(sx, (double)r));
}

// y sweep, LDS-staged; it runs before the x sweep of the stage.  One
// workgroup = 4 wavefronts = 4 adjacent columns x one run of 60 cells
// (line_tile).  The stencil inputs of the 68 cells from 4 before the run to 4
// after it, of the 4 columns, are loaded cooperatively (4 consecutive threads
// read 4 consecutive doubles of a row) into LDS, column-major; each wavefront
// then runs the per-lane computation on its column from LDS; its fluxes and
// face parts go back through LDS, where coalesced threads form the y
// divergence, scale it by dt/dy and write.  Same arithmetic as a direct
// per-lane sweep: bit-identical.
constexpr int YC = 4;          // columns per workgroup
constexpr int YR = WAVE + 4;   // stencil rows of a run
constexpr int YRP = 72;        // LDS column length: 4 columns x 8 rows fall on 32 different 8-byte banks

//
// One kernel serves a single domain (BATCH false) and a batch of domains
// (BATCH true), as the x sweep below; with the body as a device function
// called from thin kernels the FP64 HLLD / ODR 4 instance compiled to 250
// VGPRs (2 waves per SIMD) instead of 163 (3 waves).
// FMA: a tag (0 or 1) naming the build of the instantiation: the FP64
// sweeps built with FMA contraction (qas_fma64.hip) are the same template
// under FMA = 1, so their kernel symbols differ from the bit-exact ones.
// Registers: FP64 keeps the stencil in registers (HLLD 146 VGPRs, 3 waves per
// SIMD), except the batch's HLLD instance of ODR 4, whose characteristic fields
// read it from LDS again (126 VGPRs, 4 waves per SIMD: 24 domains 228 -> 220 us
// a launch; one 64^2 domain, a single round of wavefronts, took 11.5 us that
// way against 10.6).  At ODR 3 that form spills 76 bytes per lane (24 domains
// 256 us, in registers 210); at ODR 1 and 2 the two take the same time.  FP32
// tiles hold FP32 values, read from LDS (113 VGPRs).
template <int RMN, int ODR, typename T, bool BATCH, bool GRAV = false, int FMA = 0>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? (RMN >= 2 ? 3 : 4) : (BATCH && RMN == 1 && ODR == 4 ? 4 : 3)) void k_sweep2d_y(
    StagePtrs p_arg, Geo g_arg, BcFlags bc_arg, double gam, int bundle_arg, const BatchInst* I, const int* off,
    int ninst, int stage)
{
  StagePtrs p;
  Geo g;
  BcFlags bc;
  int L, bundle;
  if constexpr (BATCH) {
    const int b = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int i = batch_find(off, ninst, b);
    p = I[i].st[stage];
    g = I[i].g;
    bc = I[i].bc;
    bundle = I[i].bundle;
    L = b - off[i];
  } else {
    p = p_arg;
    g = g_arg;
    bc = bc_arg;
    bundle = bundle_arg;
    L = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  }
  __shared__ T sh[9][YC][YRP];  // ro vy vz vx bz cx pr cy by
  __shared__ T so[8][YC][YRP];  // 6 fluxes, upwind and central B-flux parts
  __shared__ T sv[RMN >= 2 ? 2 : 1][RMN >= 2 ? YRP : 1];  // vx of the columns left and right of the tile
  const int ncg = (g.nx + YC - 1) / YC;
  const int n = g.ny;
  if (L >= line_tiles(ncg, n, bundle)) return;  // whole workgroup
  const LineTile tl = line_tile(L, ncg, n, bundle);
  const long long sy = g.sy;
  // a tile of interior cells only skips the ghost-index maps (uniform)
  const bool inner = (tl.col * YC >= NG) && (tl.col * YC + YC - 1 <= g.nx - NG - 1) && (tl.row - 4 >= NG) &&
                     (tl.row + YR - 5 <= n - NG - 1);
  {
    // Staging computes the primitives of the tile's cells from the stage
    // input state (prim2d_cell, FP64) and rounds them once to the sweep
    // precision T.  The run's own cells are also stored for the x sweep, so
    // every cell of the domain is written by exactly one workgroup.
    for (int e = threadIdx.x; e < YC * YR; e += blockDim.x) {
      const int c = e % YC, r = e / YC;
      int cg, row;
      line_cell(tl, n, r - 4, cg, row);
      const int colu = cg * YC + c;
      const int col = colu > g.nx - 1 ? g.nx - 1 : colu;
      const long long a = sy * row + col;
      const Prim2d q = inner ? prim2d_cell<ODR, GRAV, true>(p, g, bc, gam, col, row, a)
                             : prim2d_cell<ODR, GRAV, false>(p, g, bc, gam, col, row, a);
      const T vx = (T)q.vx, vy = (T)q.vy, vz = (T)q.vz, pr = (T)q.pr, cx = (T)q.cx, cy = (T)q.cy;
      sh[0][c][r] = (T)G(p.in[0])[a];
      sh[1][c][r] = vy;
      sh[2][c][r] = vz;
      sh[3][c][r] = vx;
      sh[4][c][r] = (T)G(p.in[6])[a];
      sh[5][c][r] = cx;
      sh[6][c][r] = pr;
      sh[7][c][r] = cy;
      sh[8][c][r] = (T)G(p.in[5])[a];
      if (colu < g.nx && r - 4 >= tl.lo && r - 4 < tl.hi) {
        G(reinterpret_cast<T*>(p.vx))[a] = vx;
        G(reinterpret_cast<T*>(p.vy))[a] = vy;
        G(reinterpret_cast<T*>(p.vz))[a] = vz;
        G(reinterpret_cast<T*>(p.pr))[a] = pr;
        G(reinterpret_cast<T*>(p.cx))[a] = cx;
        G(reinterpret_cast<T*>(p.cy))[a] = cy;
        if constexpr (GRAV) p.enrt[a] = q.enrt;
      }
    }
    if constexpr (RMN >= 2) {
      if (inner && threadIdx.x < 2 * YR) {  // (which other workgroups of this launch store: from the state)
        const int side = threadIdx.x < YR ? 0 : 1, r = (int)threadIdx.x - side * YR;
        const VelOf<T> vxs{p.in[1], p.in[0]};
        sv[side][r] = vxs[sy * (tl.row + r - 4) + tl.col * YC + (side ? YC : -1)];
      }
    }
  }
  __syncthreads();
  const int w = threadIdx.x / WAVE;
  const int lane = threadIdx.x & (WAVE - 1);
  const int rb = lane + 2;  // this lane's cell in the tile
  // the stencil in registers, or left in LDS for each characteristic field to
  // read its part
  constexpr bool IN_LDS = sizeof(T) == 4 || (BATCH && RMN == 1 && ODR == 4);
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
  // B-flux face states first, then the characteristic reconstruction
  T ql, qr;
  {
    T pp[5], qq[5];
#pragma unroll
    for (int m = 0; m < 5; m++) {
      pp[m] = s(5, m) * s(1, m);  // cx * vy
      qq[m] = s(3, m);            // vx
    }
    lr_fb<ODR>(pp, qq, sh[8][w][rb], sh[8][w][rb + 1], ql, qr);
  }
  s.again();
  T vl[7], vr[7];
  lrstate_of<ODR, T, 0, true, (sizeof(T) == 8 || RMN >= 2)>(s, sh[7][w][rb], (T)gam, vl, vr);
  T Lf[7], Rf[7], F[7];
#pragma unroll
  for (int k = 0; k < 7; k++) {
    Lf[k] = __shfl_up(vl[k], 1, WAVE);
    Rf[k] = vr[k];
  }
  const T qlf = __shfl_up(ql, 1, WAVE);
  const T bnf = sh[8][w][rb];  // (both sides of the face share it)
  T dv0 = T(0.0), dv1 = T(0.0);
  // the lane's column and face where global arrays are read (lanes past the
  // domain: some cell of it)
  int lc = 0, q = 0, sf = 3;
  if constexpr (RMN >= 2 || GRAV) {
    int cg;
    line_cell(tl, n, lane - 2, cg, q);
    sf = q < 3 ? 3 : (q > n - 3 ? n - 3 : q);
    lc = cg * YC + w > g.nx - 1 ? g.nx - 1 : cg * YC + w;
  }
  if constexpr (RMN >= 2) {
    dv0 = sh[1][w][rb] - sh[1][w][rb - 1];
    // the transverse sensor of this lane's cell; the other one of its face is
    // the lane before's.  An interior tile has vx of the neighbouring columns
    // in LDS; elsewhere it comes from the state through the index maps, with
    // the primitive's own expression and rounding
    T dvc;
    if (inner) {
      const T v = sh[3][w][rb];
      const T vm = w > 0 ? sh[3][w > 0 ? w - 1 : 0][rb] : sv[0][rb], vp = w < YC - 1 ? sh[3][w < YC - 1 ? w + 1 : 0][rb] : sv[1][rb];
      dvc = tmin(vp - v, v - vm);
    } else {
      const VelOf<T> vxs{p.in[1], p.in[0]};
      dvc = (T)dv_at<0>(vxs, lc, q, g, bc);
    }
    dv1 = tmin((T)__shfl_up(dvc, 1, WAVE), dvc);
  }
  riemann<RMN>(Lf, Rf, bnf, (T)gam, dv0, dv1, F);
  const T fc = T(0.5) * (qlf + qr);
  const T fbu = F[5] - fc;
  // y: (F0, F3, F1, F2, F4, F6) feed (ro, mx, my, mz, bz, en)
  if constexpr (GRAV)  // work done by gravity (2D/SERIAL/RTI/mhd2d_solve.cpp:305)
    F[6] += F[0] * 0.5 * (p.phi[lc + sy * (sf - 1)] + p.phi[lc + sy * sf]);
  const int fid[6] = {0, 3, 1, 2, 4, 6};
#pragma unroll
  for (int v = 0; v < 6; v++) so[v][w][lane] = F[fid[v]];
  so[6][w][lane] = fbu;
  so[7][w][lane] = fc;
  __syncthreads();
  // coalesced write-back: thread -> (column c, lane r) of the 4 x 64 tile
  {
    const int c = threadIdx.x % YC, r = threadIdx.x / YC;
    int cg, row;
    line_cell(tl, n, r - 2, cg, row);
    const int i = cg * YC + c;
    const bool own = (r >= 2) && (r - 2 < tl.hi) && (r < 2 + SEG) && (row >= 3) && (row <= n - 3) && (i < g.nx);
    if (own) {
      const long long a = sy * row + i;
      store_as<T>(p.emf[4], a, so[6][c][r]);
      store_as<T>(p.emf[5], a, so[7][c][r]);
      const bool upd = (row >= NG) && (row <= n - NG - 1) && (i >= NG) && (i <= g.nx - NG - 1);
      if (upd) {
        // dt/dy * Dy of (ro, mx, my, mz, bz, en); the x sweep, which runs
        // next, subtracts it in the stage sum
        const double dtdy = G(p.dt)[0] / g.dy;
#pragma unroll
        for (int v = 0; v < 6; v++)
          store_as<T>(p.acc[v], a, dtdy * dfc<ODR>((double)so[v][c][r - 1], (double)so[v][c][r], (double)so[v][c][r + 1],
                                               (double)so[v][c][r + 2]));
      }
    }
  }
}

// ------------------------------------------------------------------ x sweep
// x faces of every row; it runs after the y sweep and applies the RK stage
// sum.  The cells of the domain in memory order are cut into runs of
// (workgroup size - 4) whatever row they fall in; lane t of a workgroup takes
// cell t - 2 of its run, and left states and fluxes pass between its lanes
// through LDS.  Against one run of 60 faces per wavefront and row, which
// handed them over by shuffles, that is 9 % fewer wavefronts at 1024^2 (28 %
// at 128^2): one halo for the workgroup instead of one per wavefront, and no
// partly empty wavefront at the end of each row.
// One kernel serves a single domain (BATCH false: the stage descriptor is the
// kernel argument) and a batch of domains (BATCH true: the instance table, as
// kb_* kernels).
// FP32 stages the stencil inputs in LDS too (one load per value and cell) and
// each characteristic field reads its part again: 116 VGPRs and 35 fewer loads
// a lane, MLAU at 2048^2 247 -> 202 us.  FP64 loads its stencil straight into
// registers: from LDS it gained nothing (142 VGPRs as before, 83.3 us against
// 82.2 at 1024^2; held to 4 waves per SIMD it spilled, 105 us).  3 waves per
// SIMD for every FP64 instance: Roe and MLAU with gravity at ODR 4 spill 20
// bytes per lane for it, 512 x 1024 50.5 us against 53.4 in 2 waves without.
// LDS per lane: the cell's 7 values (then its 6 fluxes) and, apart from them,
// 8 face values and the sensor; odd strides, so that 64 lanes fall on different banks.
constexpr int XS = 7, XL = 9;
template <typename T>
constexpr unsigned x_lds_bytes(int nb) { return (unsigned)((XS * (nb + HALO) + XL * nb) * sizeof(T)); }

// the run of a workgroup: cells [first, first + own) of the array, of which
// this thread has cell a (clamped into the array), at (i, row)
struct XCell {
  long long a;
  int i, row;
  bool own;  // the thread's own cell, not a halo lane
};
__device__ __forceinline__ XCell x_cell(int blk, int nx, long long nd)
{
  const int own = (int)blockDim.x - HALO;
  const long long first = (long long)blk * own;
  const int t = (int)threadIdx.x;
  XCell c;
  const unsigned row0 = (unsigned)first / (unsigned)nx;
  c.row = (int)row0;
  c.i = (int)(first - (long long)row0 * nx) + t - 2;
  c.a = first + t - 2;
  c.own = t >= 2 && t < 2 + own && c.a < nd;
  if (c.a < 0) { c.a = 0; c.i = 0; }
  while (c.i >= nx) { c.i -= nx; c.row++; }
  while (c.i < 0) { c.i += nx; c.row--; }
  if (c.a >= nd) { c.a = nd - 1; c.i = nx - 1; c.row = (int)((unsigned)(nd - 1) / (unsigned)nx); }
  return c;
}

template <int RMN, int ODR, typename T, bool BATCH, bool GRAV = false, int FMA = 0>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? (RMN >= 2 ? 4 : 1) : 3) void k_sweep2d(StagePtrs p_arg, Geo g_arg, BcFlags bc_arg, double gam,
                                                 int, const BatchInst* I, const int* off, int ninst, int stage)
{
  StagePtrs p;
  Geo g;
  BcFlags bc;
  int blk;
  if constexpr (BATCH) {
    const int b = (int)blockIdx.x;
    const int i = batch_find(off, ninst, b);
    p = I[i].st[stage];
    g = I[i].g;
    bc = I[i].bc;
    blk = b - off[i];
  } else {
    p = p_arg;
    g = g_arg;
    bc = bc_arg;
    blk = (int)blockIdx.x;
  }
  extern __shared__ double x_lds[];
  const int nb = (int)blockDim.x;
  T* const xs = reinterpret_cast<T*>(x_lds) + XS * ((int)threadIdx.x + 2);               // this lane's cell
  T* const xl = reinterpret_cast<T*>(x_lds) + XS * (nb + HALO) + XL * (int)threadIdx.x;  // its face values
  const int n = g.nx;
  const XCell cell = x_cell(blk, n, g.nd);
  const int q = cell.i, line = cell.row;
  const long long base = cell.a - q;  // the row's first cell

  // primitive stencil, cyclic order (vn, vt, vu), (bt, bu); bt = cy is the
  // tangential component that pairs with this sweep, bu = bz.  (A lane whose
  // stencil would cross the end of its row takes the row's last full one or
  // whatever is next in memory; nothing uses what it computes.)
  const PrimView<T> pv = prim_view<T>(p);
  const auto bf = G(p.in[4]);      // staggered normal B
  auto load = [&](int k, long long a) -> T {
    switch (k) {
      case 0: return (T)G(p.in[0])[a];
      case 1: return G(pv.vx)[a];
      case 2: return G(pv.vy)[a];
      case 3: return G(pv.vz)[a];
      case 4: return G(pv.cy)[a];
      case 5: return (T)G(p.in[6])[a];
      default: return G(pv.pr)[a];
    }
  };
  T sr[7][5];
  if constexpr (sizeof(T) == 8) {
    const long long sc = base + (q < 2 ? 2 : (q > n - 3 ? n - 3 : q));
#pragma unroll
    for (int m = 0; m < 5; m++)
#pragma unroll
      for (int k = 0; k < 7; k++) sr[k][m] = load(k, sc + (m - 2));
  } else {
#pragma unroll
    for (int k = 0; k < 7; k++) xs[k] = load(k, cell.a);
    if (threadIdx.x < HALO) {  // the 2 cells before the first lane's and the 2 after the last one's
      const int d = threadIdx.x < 2 ? (int)threadIdx.x - 2 : nb + (int)threadIdx.x - 2;
      long long a = (long long)blk * (nb - HALO) - 2 + d;
      a = a < 0 ? 0 : (a > g.nd - 1 ? g.nd - 1 : a);
#pragma unroll
      for (int k = 0; k < 7; k++) reinterpret_cast<T*>(x_lds)[XS * (d + 2) + k] = load(k, a);
    }
  }
  const T cn = (T)G(pv.cx)[cell.a], bm = (T)bf[cell.a], bp = (T)bf[cell.a + 1 < g.nd ? cell.a + 1 : cell.a];
  if constexpr (sizeof(T) == 4) __syncthreads();
  const auto s = [&]() {
    if constexpr (sizeof(T) == 8) return RegStencil<T>{sr};
    else return LdsStencil<T, T, 1, XS>{xs};
  }();
  // B-flux face states (mhd_lr_fb): b_t v_n - b_n v_t
  T ql, qr;
  {
    T pp[5], qq[5];
#pragma unroll
    for (int m = 0; m < 5; m++) {
      pp[m] = s(4, m) * s(1, m);
      qq[m] = s(2, m);
    }
    lr_fb<ODR>(pp, qq, bm, bp, ql, qr);
  }
  const T vnf = s(1, 2), vnb = s(1, 1);  // of the face's two cells
  s.again();
  T vl[7], vr[7];
  lrstate_of<ODR, T, 0, true, std::is_same<T, double>::value>(s, cn, (T)gam, vl, vr);

  // flux at face q (between q-1 and q): left state from the lane before
  // (lane 0 has none: its flux is not used)
#pragma unroll
  for (int k = 0; k < 7; k++) xl[k] = vl[k];
  xl[7] = ql;
  // the transverse sensor of this lane's cell, handed over too
  T dvc = T(0.0);
  if constexpr (RMN >= 2) {
    const auto vy = G(pv.vy);
    if (__all((q >= NG) & (q <= n - NG - 1) & (line >= NG) & (line <= g.ny - NG - 1))) {
      const T v = s(2, 2);
      dvc = tmin(vy[cell.a + g.sy] - v, v - vy[cell.a - g.sy]);
    } else {
      dvc = (T)dv_at<1>(pv.vy, q, line, g, bc);
    }
    xl[8] = dvc;
  }
  __syncthreads();
  const T* const xb = threadIdx.x > 0 ? xl - XL : xl;
  T L[7], F[7];
#pragma unroll
  for (int k = 0; k < 7; k++) L[k] = xb[k];
  const T qlf = xb[7];
  const int qf = q < 3 ? 3 : (q > n - 3 ? n - 3 : q);
  const long long sf = base + qf;  // face index (clamped)
  const T bnf = bm;                // (both sides of the face share it)
  T dv0 = T(0.0), dv1 = T(0.0);
  if constexpr (RMN >= 2) {
    dv0 = vnf - vnb;
    dv1 = tmin(xb[8], dvc);
  }
  riemann<RMN>(L, vr, bnf, (T)gam, dv0, dv1, F);
  const T fc = T(0.5) * (qlf + qr);
  const T fbu = F[4] - fc;  // split of the By flux

  const bool own = cell.own && (q >= 3) && (q <= n - 3);
  if (own) {
    store_as<T>(p.emf[0], cell.a, (double)fbu);
    store_as<T>(p.emf[1], cell.a, (double)fc);
  }

  // flux divergence of ro, mx, my, mz, bz, en at cell q: faces q-1 .. q+2,
  // (F0, F1, F2, F3, F5, F6), differenced in FP64 in both precisions
  if constexpr (GRAV) F[6] += F[0] * 0.5 * (p.phi[sf - 1] + p.phi[sf]);  // work done by gravity (RTI:197)
  const int fid[6] = {0, 1, 2, 3, 5, 6};
#pragma unroll
  for (int v = 0; v < 6; v++) xs[v] = F[fid[v]];  // (every lane has read its stencil)
  __syncthreads();
  const bool upd = own && (q >= NG) && (q <= n - NG - 1) && (line >= NG) && (line <= g.ny - NG - 1);
  if (!upd) return;
  // the y sweep ran first and left acc = dt/dy * Dy; the stage sum
  // u = a u0 + b (u + ((-dt/dx Dx) - dt/dy Dy)) is the reference's
  // expression in its order (mhd2d_solve.cpp:199, 341-358)
  const long long c = cell.a;
  const double dtdx = G(p.dt)[0] / g.dx;
  const int vid[6] = {0, 1, 2, 3, 6, 7};
  double un[6];
#pragma unroll
  for (int v = 0; v < 6; v++) {
    const int m = vid[v];
    const double du = dfc<ODR>((double)xs[v - XS], (double)F[fid[v]], (double)xs[v + XS], (double)xs[v + 2 * XS]);
    un[v] = rk_upd(G(p.in[m])[c], G(p.u0[m])[c], (-dtdx * du) - load_as<T>(p.acc[v], c), p.a, p.b);
  }
  if constexpr (GRAV) {
    // gravity on the momentum with the updated density (RTI/mhd2d_solve.cpp:361-362)
    const double dtdy = *p.dt / g.dy;
    un[1] += -p.b * un[0] * 0.5 * (p.phi[c + 1] - p.phi[c - 1]) * dtdx;
    un[2] += -p.b * un[0] * 0.5 * (p.phi[c + g.sy] - p.phi[c - g.sy]) * dtdy;
  }
#pragma unroll
  for (int v = 0; v < 6; v++) G(p.out[vid[v]])[c] = un[v];
}

// kernel tables: y sweep and x sweep (single domain or batch)
template <typename T, int FMA = 0>
xsweep2d_fn pick_ysweep2d_t(int rmn, int odr, bool batch)
{
#define QAS_S(R, O) \
  if (rmn == R && odr == O) return batch ? k_sweep2d_y<R, O, T, true, false, FMA> : k_sweep2d_y<R, O, T, false, false, FMA>;
  QAS_S(0, 1) QAS_S(0, 2) QAS_S(0, 3) QAS_S(0, 4)
  QAS_S(1, 1) QAS_S(1, 2) QAS_S(1, 3) QAS_S(1, 4)
  QAS_S(2, 1) QAS_S(2, 2) QAS_S(2, 3) QAS_S(2, 4)
  QAS_S(3, 1) QAS_S(3, 2) QAS_S(3, 3) QAS_S(3, 4)
#undef QAS_S
  return nullptr;
}

template <typename T, int FMA = 0>
xsweep2d_fn pick_xsweep2d_t(int rmn, int odr, bool batch)
{
#define QAS_S(R, O) \
  if (rmn == R && odr == O) return batch ? k_sweep2d<R, O, T, true, false, FMA> : k_sweep2d<R, O, T, false, false, FMA>;
  QAS_S(0, 1) QAS_S(0, 2) QAS_S(0, 3) QAS_S(0, 4)
  QAS_S(1, 1) QAS_S(1, 2) QAS_S(1, 3) QAS_S(1, 4)
  QAS_S(2, 1) QAS_S(2, 2) QAS_S(2, 3) QAS_S(2, 4)
  QAS_S(3, 1) QAS_S(3, 2) QAS_S(3, 3) QAS_S(3, 4)
#undef QAS_S
  return nullptr;
}

}  // namespace qas
