// A whole WENO or MUSCL stage in one kernel for tables of 1D problems: boxes
// 4 x 4 cells across, periodic in y and z (Sod tubes, Riemann sweeps).
//
// The directional passes (dir_flux.hip) read the state once per direction,
// convert it again each time and carry the sum of the earlier passes through
// HBM: 360 B per cell and stage against 120, and on a small tube nine launches
// per step that each last one workgroup's latency.  Here the 16 cells of a
// cross-section are one 16-lane row of a wave (lane = y + 4 z), so the y and z
// neighbours of a cell are lanes of its own row, reached by DPP (quad
// permutations and row rotations), and only the x pencils go through LDS.  The
// faces, their sum x + y + z per cell, the source-free stage combination and
// every operation of a face are the passes'.
//
// A brick is up to NX cells along x; thread (xi, lane) owns cell xi and the
// face below it.  Few bricks (a tube alone on the chip) are bound by the
// latency of one thread's faces: the split kernels give every wave one
// direction (MUSCL) or one component of one direction (WENO) of a short
// brick.
//
// Measured (MI355X, us a stage, passes -> this): batch of 512 problems (8.65M
// cells) WENO 1240 -> 889, of 128 problems (1.15M cells) MUSCL 184 -> 129; Sod
// tube 256 x 4 x 4 WENO 25 -> 7.7, MUSCL 24 -> 9.2 (86 split bricks).  Bound
// by FP64 issue (divisions and square roots) on the batches, by one brick's
// latency on a tube.
#include "cns_point.h"
#include "kernels.h"

namespace amr {

namespace {

constexpr int TR = 16;  // rows of a tube: lane = y + 4 z

// DPP controls: the value of the row TR-lane that lies m cells on in y or z
// (periodic over 4)
template <int D, int M>
__device__ __forceinline__ double row_shift(double v) {
  constexpr int m = (M + 4) & 3;
  if constexpr (m == 0) {
    return v;
  } else {
    constexpr int yq = m == 1 ? 0x39 : (m == 2 ? 0x4E : 0x93);  // quad_perm (1,2,3,0), (2,3,0,1), (3,0,1,2)
    constexpr int zr = 0x120 + 16 - 4 * m;                       // row_ror: lane i takes lane i + 4 m
    constexpr int ctrl = D == 1 ? yq : zr;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
  }
}

// The conserved state of cell x of row r of brick W's box (x up to NGHOST
// cells beyond the box: periodic images of the box itself, or the side
// tables' neighbour cell or boundary rule; clamped there past the last ghost
// cell, for lanes beyond a short brick).
__device__ __forceinline__ void tube_cell(const TubeBrick& W, const BoxDev& bx, const Fab& S, const XSide* xs,
                                          const Fab* __restrict__ sinf, int x, int r, double u[5]) {
  const int j = bx.lo[1] + (r & 3), k = bx.lo[2] + (r >> 2);
  if (W.wrap > 0) {
    x = bx.lo[0] + ((x - bx.lo[0]) % W.wrap + W.wrap) % W.wrap;
  } else {
    x = min(x, bx.hi[0] + NGHOST);
    if (x < bx.lo[0] || x > bx.hi[0]) {
      const int side = x > bx.hi[0] ? 1 : 0;
      const XSide X = xs[2 * W.box + side];
      if (X.kind == 1) {
        const Fab F = sinf[X.src];
#pragma unroll
        for (int n = 0; n < 5; ++n) u[n] = F(x + X.shift, j, k, n);
        return;
      }
      // k_fill_bc's rule (AMReX foextrap / reflect_even / reflect_odd)
#pragma unroll
      for (int n = 0; n < 5; ++n) {
        const int ty = X.type[n];
        const double v = S(ty == 2 ? X.bnd : (side == 0 ? 2 * X.bnd - 1 - x : 2 * X.bnd + 1 - x), j, k, n);
        u[n] = ty == 4 ? -v : v;
      }
      return;
    }
  }
#pragma unroll
  for (int n = 0; n < 5; ++n) u[n] = S(x, j, k, n);
}

// Stage combination of a cell's dSdt L (source and body force as the last
// directional pass adds them).
__device__ __forceinline__ void tube_store(const StageArgs& sa, const StageCoef& sc, int b, const Fab& O, int i, int j,
                                           int k, int n, double L, double s1, double u, double rho, double mx) {
  if (sa.src) L = L + sa.src[b](i, j, k, n);  // user_source, CNS_advance.cpp:397-407
  if (sa.bfx != 0.0 && n == UMX) L = L + rho * sa.bfx;
  if (sa.bfx != 0.0 && n == UET) L = L + mx * sa.bfx;
  O(i, j, k, n) = sc.mode == 2 ? L : stage_combine(sc, s1, u, L);
}

// ---------------------------------------------------------------- WENO
// Per cell: conserved state, pressure, velocity and wave speed per direction
// (High_resolution.h:83-121).
struct WCell {
  double u[5], P, vel[3], lam[3];
};
__device__ __forceinline__ void weno_cell(const double u[5], const Closures& c, WCell& w) {
  const double rho = u[URHO];
  const double rhoinv = 1.0 / rho;
  const double rhoekin = 0.5 * rhoinv * (u[UMX] * u[UMX] + u[UMY] * u[UMY] + u[UMZ] * u[UMZ]);
  const double rhoeint = u[UET] - rhoekin;
  w.P = c.gm1 * rhoeint;
  const double cs = sqrt(c.gamma * w.P * rhoinv);
#pragma unroll
  for (int n = 0; n < 5; ++n) w.u[n] = u[n];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    w.vel[d] = u[UMX + d] * rhoinv;
    w.lam[d] = fabs(dmax(dmax(w.vel[d] + cs, w.vel[d] - cs), w.vel[d]));
  }
}

// Half of the flux of component n along D (the split fluxes' half is exact)
__device__ __forceinline__ double half_flux(int D, int n, double un, double md, double E, double P, double hud) {
  if (n == URHO) return 0.5 * md;
  if (n == UET) return (E + P) * hud;
  return n == 1 + D ? un * hud + 0.5 * P : un * hud;
}

// numericalflux_globallaxsplit (High_resolution.h:162-246) from the six half
// fluxes Pf and states U of the stencil and half the wave-speed maximum.
__device__ __forceinline__ double weno_split(const double Pf[6], const double U[6], double hme) {
  double df[6];
#pragma unroll
  for (int o = 0; o < 6; ++o) df[o] = hme * U[o];
  bool ok = true;
  double f = weno5js_fast(Pf[0] + df[0], Pf[1] + df[1], Pf[2] + df[2], Pf[3] + df[3], Pf[4] + df[4], ok);
  f += weno5js_fast(Pf[5] - df[5], Pf[4] - df[4], Pf[3] - df[3], Pf[2] - df[2], Pf[1] - df[1], ok);
  if (!ok) {
    f = weno5js(Pf[0] + df[0], Pf[1] + df[1], Pf[2] + df[2], Pf[3] + df[3], Pf[4] + df[4]);
    f += weno5js(Pf[5] - df[5], Pf[4] - df[4], Pf[3] - df[3], Pf[2] - df[2], Pf[1] - df[1]);
  }
  return f;
}

// dxi (F(below) - F(above)) of component n along D (1 y, 2 z) for the lane's
// cell: the stencil -3 .. 2 holds four distinct cells of the periodic row.
template <int D, int N>
__device__ __forceinline__ double weno_row_diff(const WCell& w, double hme, double dxi) {
  const double p = half_flux(D, N, w.u[N], w.u[1 + D], w.u[UET], w.P, 0.5 * w.vel[D]);
  const double p1 = row_shift<D, 1>(p), p2 = row_shift<D, 2>(p), pm = row_shift<D, -1>(p);
  const double u1 = row_shift<D, 1>(w.u[N]), u2 = row_shift<D, 2>(w.u[N]), um = row_shift<D, -1>(w.u[N]);
  const double Pf[6] = {p1, p2, pm, p, p1, p2}, U[6] = {u1, u2, um, w.u[N], u1, u2};
  const double f = weno_split(Pf, U, hme);
  return dxi * (f - row_shift<D, 1>(f));
}
template <int D>
__device__ __forceinline__ void weno_row(const WCell& w, double dxi, double t[5]) {
  // the maximum over the stencil's cells in its order (repeats change nothing)
  double me = row_shift<D, 1>(w.lam[D]);
  me = dmax(me, row_shift<D, 2>(w.lam[D]));
  me = dmax(me, row_shift<D, -1>(w.lam[D]));
  me = dmax(me, w.lam[D]);
  const double hme = 0.5 * me;
  // (one component at a time, as in the directional passes)
  t[0] = weno_row_diff<D, 0>(w, hme, dxi);
  __builtin_amdgcn_sched_barrier(0);
  t[1] = weno_row_diff<D, 1>(w, hme, dxi);
  __builtin_amdgcn_sched_barrier(0);
  t[2] = weno_row_diff<D, 2>(w, hme, dxi);
  __builtin_amdgcn_sched_barrier(0);
  t[3] = weno_row_diff<D, 3>(w, hme, dxi);
  __builtin_amdgcn_sched_barrier(0);
  t[4] = weno_row_diff<D, 4>(w, hme, dxi);
  __builtin_amdgcn_sched_barrier(0);
}

template <int NX>
__global__ void __launch_bounds__((NX + 1) * TR, 4)
k_weno_tube(const TubeBrick* __restrict__ bricks, const BoxDev* __restrict__ boxes, Closures c, StageArgs sa,
            const Fab* __restrict__ sinf, const Fab* __restrict__ s1f, const Fab* __restrict__ outf,
            const XSide* __restrict__ xs) {
  constexpr int NT = (NX + 1) * TR, NC = (NX + 6) * TR;  // cell column xi at (xi + 3) * TR
  __shared__ double sv[8][NC];                           // conserved state, x velocity, pressure, x wave speed
  __shared__ double sF[5][NT];
  const TubeBrick W = bricks[blockIdx.x];
  if (W.nx <= 0 || !box_active(sa, W.box)) return;  // uniform
  const BoxDev bx = boxes[W.box];
  const Fab S = sinf[W.box];
  const int t = threadIdx.x, r = t & (TR - 1), xi = t / TR;
  auto put = [&](int l, const WCell& w) {
#pragma unroll
    for (int n = 0; n < 5; ++n) sv[n][l] = w.u[n];
    sv[5][l] = w.vel[0];
    sv[6][l] = w.P;
    sv[7][l] = w.lam[0];
  };
  WCell w;
  {
    double u[5], h[5];
    tube_cell(W, bx, S, xs, sinf, W.x0 + xi, r, u);
    // the five columns beyond the threads' own
    for (int q = t; q < 5 * TR; q += NT) {
      const int hc = q / TR < 3 ? q / TR : NX + 1 + q / TR;
      WCell g;
      tube_cell(W, bx, S, xs, sinf, W.x0 + hc - 3, r, h);
      weno_cell(h, c, g);
      put(hc * TR + r, g);
    }
    weno_cell(u, c, w);
    put((xi + 3) * TR + r, w);
  }
  double ty[5], tz[5];
  weno_row<1>(w, bx.dxi[1], ty);
  weno_row<2>(w, bx.dxi[2], tz);
  __syncthreads();
  // x faces: face xi below cell xi, stencil columns xi .. xi + 5
  double F[5];
  {
    const int l0 = xi * TR + r;
    double me = sv[7][l0];
#pragma unroll
    for (int o = 1; o < 6; ++o) me = dmax(me, sv[7][l0 + o * TR]);
    const double hme = 0.5 * me;
#pragma unroll
    for (int n = 0; n < 5; ++n) {
      double Pf[6], U[6];
#pragma unroll
      for (int o = 0; o < 6; ++o) {
        const int l = l0 + o * TR;
        U[o] = sv[n][l];
        Pf[o] = half_flux(0, n, U[o], sv[1][l], sv[4][l], sv[6][l], 0.5 * sv[5][l]);
      }
      F[n] = weno_split(Pf, U, hme);
      sF[n][t] = F[n];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  if (xi >= W.nx) return;
  const StageCoef sc = box_stage(sa, W.box);
  const bool use_s1 = sc.mode != 2 && sc.a != 0.0;
  const Fab O = outf[W.box];
  const int i = W.x0 + xi, j = bx.lo[1] + (r & 3), k = bx.lo[2] + (r >> 2);
  const int l = (xi + 3) * TR + r;
#pragma unroll
  for (int n = 0; n < 5; ++n) {
    const double L = (bx.dxi[0] * (F[n] - sF[n][t + TR]) + ty[n]) + tz[n];
    tube_store(sa, sc, W.box, O, i, j, k, n, L, use_s1 ? s1f[W.box](i, j, k, n) : 0.0, sv[n][l], sv[URHO][l],
               sv[UMX][l]);
  }
}

// A short brick over 15 waves: wave w forms component w % 5 of the faces along
// direction w / 5, all stencils from LDS.
constexpr int SX = 3;  // cells of a split brick
__global__ void __launch_bounds__(15 * 64)
k_weno_tube_split(const TubeBrick* __restrict__ bricks, const BoxDev* __restrict__ boxes, Closures c, StageArgs sa,
                  const Fab* __restrict__ sinf, const Fab* __restrict__ s1f, const Fab* __restrict__ outf,
                  const XSide* __restrict__ xs) {
  constexpr int NC = (SX + 6) * TR;
  __shared__ double su[5][NC], sp[NC], svel[3][NC], slam[3][NC];
  __shared__ double sF[15][(SX + 1) * TR];
  const TubeBrick W = bricks[blockIdx.x];
  if (W.nx <= 0 || !box_active(sa, W.box)) return;  // uniform
  const BoxDev bx = boxes[W.box];
  const int t = threadIdx.x;
  const StageCoef sc = box_stage(sa, W.box);
  const bool use_s1 = sc.mode != 2 && sc.a != 0.0;
  // thread t < 240 finishes component t / 48 of cell t % 48
  const int fn = t / (SX * TR), fc = t % (SX * TR), fr = fc & (TR - 1);
  const int i = W.x0 + fc / TR, j = bx.lo[1] + (fr & 3), k = bx.lo[2] + (fr >> 2);
  const bool fin = fn < 5 && fc / TR < W.nx;
  double s1 = 0.0;
  if (fin && use_s1) s1 = s1f[W.box](i, j, k, fn);
  if (t < NC) {
    double u[5];
    tube_cell(W, bx, sinf[W.box], xs, sinf, W.x0 + t / TR - 3, t & (TR - 1), u);
    WCell w;
    weno_cell(u, c, w);
#pragma unroll
    for (int n = 0; n < 5; ++n) su[n][t] = w.u[n];
    sp[t] = w.P;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      svel[d][t] = w.vel[d];
      slam[d][t] = w.lam[d];
    }
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6), D = wv / 5, n = wv % 5;
  const int lane = t & 63, r = lane & (TR - 1), xi = lane / TR;
  {
    double Pf[6], U[6], me = 0.0;
#pragma unroll
    for (int o = 0; o < 6; ++o) {
      int l;
      if (D == 0) l = (xi + o) * TR + r;
      else if (D == 1) l = (xi + 3) * TR + (r & 12) + ((r + o + 1) & 3);
      else l = (xi + 3) * TR + ((r + 4 * (o + 1)) & 15);
      me = o == 0 ? slam[D][l] : dmax(me, slam[D][l]);
      U[o] = su[n][l];
      Pf[o] = half_flux(D, n, U[o], su[1 + D][l], su[UET][l], sp[l], 0.5 * svel[D][l]);
    }
    sF[wv][lane] = weno_split(Pf, U, 0.5 * me);
  }
  __syncthreads();
  if (!fin) return;
  double L = bx.dxi[0] * (sF[fn][fc] - sF[fn][fc + TR]);
  L = L + bx.dxi[1] * (sF[5 + fn][fc] - sF[5 + fn][(fc & ~3) + ((fc + 1) & 3)]);
  L = L + bx.dxi[2] * (sF[10 + fn][fc] - sF[10 + fn][(fc & ~15) + ((fc + 4) & 15)]);
  const int l = fc + 3 * TR;
  tube_store(sa, sc, W.box, outf[W.box], i, j, k, fn, L, s1, su[fn][l], su[URHO][l], su[UMX][l]);
}

// ---------------------------------------------------------------- MUSCL
// dxi (F(below) - F(above)) along D (1 y, 2 z) for the lane's cell q.
template <int D>
__device__ __forceinline__ void muscl_row(const double q[NPRIM], const Closures& c, double dxi, double t[5]) {
  double qp[NPRIM], qm[NPRIM], d[5], dm[5], F[5];
#pragma unroll
  for (int n = 0; n < NPRIM; ++n) {
    qp[n] = row_shift<D, 1>(q[n]);
    qm[n] = row_shift<D, -1>(q[n]);
  }
  auto Q = [&](int o, int comp) { return o == 0 ? q[comp] : (o == 1 ? qp[comp] : qm[comp]); };
  muscl_slopes<D>(Q, c, d);
#pragma unroll
  for (int n = 0; n < 5; ++n) dm[n] = row_shift<D, -1>(d[n]);
  auto ql = [&](int n) { return qm[n]; };
  auto dql = [&](int n) { return dm[n]; };
  auto qr = [&](int n) { return q[n]; };
  auto dqr = [&](int n) { return d[n]; };
  // the z left state's sound speed comes from T at k+1 (Riemann.h:316)
  muscl_face<D>(ql, dql, qr, dqr, D == 2 ? qp[QT] : qm[QT], c, F);
#pragma unroll
  for (int n = 0; n < 5; ++n) t[n] = dxi * (F[n] - row_shift<D, 1>(F[n]));
}

// SPLIT: three groups of NT threads, one per direction (few bricks); else
// every thread forms the faces of its cell along all three.
template <int NX, bool SPLIT>
__global__ void __launch_bounds__((NX + 1) * TR * (SPLIT ? 3 : 1))
k_muscl_tube(const TubeBrick* __restrict__ bricks, const BoxDev* __restrict__ boxes, Closures c, StageArgs sa,
             const Fab* __restrict__ sinf, const Fab* __restrict__ s1f, const Fab* __restrict__ outf,
             const XSide* __restrict__ xs) {
  constexpr int NT = (NX + 1) * TR, NC = (NX + 4) * TR;  // cell column xi at (xi + 2) * TR
  __shared__ double sq[NPRIM][NC];
  __shared__ double sd[5][NT + TR];  // x slopes of columns -1 .. NX
  __shared__ double sF[5][NT];
  __shared__ double st[SPLIT ? 10 : 1][SPLIT ? NT : 1];  // y and z terms
  const TubeBrick W = bricks[blockIdx.x];
  if (W.nx <= 0 || !box_active(sa, W.box)) return;  // uniform
  const BoxDev bx = boxes[W.box];
  const Fab S = sinf[W.box];
  const int grp = SPLIT ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
  const int t = SPLIT ? threadIdx.x % NT : threadIdx.x;
  const int r = t & (TR - 1), xi = t / TR;
  const int i = W.x0 + xi, j = bx.lo[1] + (r & 3), k = bx.lo[2] + (r >> 2);
  const StageCoef sc = box_stage(sa, W.box);
  const bool use_s1 = sc.mode != 2 && sc.a != 0.0;
  double u[5], q[NPRIM], s1[5];
  tube_cell(W, bx, S, xs, sinf, i, r, u);
  if (SPLIT && grp == 0 && use_s1 && xi < W.nx)
#pragma unroll
    for (int n = 0; n < 5; ++n) s1[n] = s1f[W.box](i, j, k, n);
  if (grp == 0)
    for (int h = t; h < 3 * TR; h += NT) {
      const int hc = h / TR < 2 ? h / TR : NX + 3;
      double v[5], p[NPRIM];
      tube_cell(W, bx, S, xs, sinf, W.x0 + hc - 2, r, v);
      cons2prim(v[0], v[1], v[2], v[3], v[4], c, p);
#pragma unroll
      for (int n = 0; n < NPRIM; ++n) sq[n][hc * TR + r] = p[n];
    }
  cons2prim(u[0], u[1], u[2], u[3], u[4], c, q);
  if (grp == 0)
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) sq[n][(xi + 2) * TR + r] = q[n];
  double ty[5], tz[5];
  if (!SPLIT || grp == 1) muscl_row<1>(q, c, bx.dxi[1], ty);
  if (!SPLIT || grp == 2) muscl_row<2>(q, c, bx.dxi[2], tz);
  if (SPLIT && grp == 1)
#pragma unroll
    for (int n = 0; n < 5; ++n) st[n][t] = ty[n];
  if (SPLIT && grp == 2)
#pragma unroll
    for (int n = 0; n < 5; ++n) st[5 + n][t] = tz[n];
  __syncthreads();
  // x slopes of columns 0 .. NX, and of column -1 on the first row of threads
  // of another group where there is one
  auto slope = [&](int col) {
    const int l = (col + 2) * TR + r;
    auto Q = [&](int o, int comp) { return sq[comp][l + o * TR]; };
    double d[5];
    muscl_slopes<0>(Q, c, d);
#pragma unroll
    for (int n = 0; n < 5; ++n) sd[n][(col + 1) * TR + r] = d[n];
  };
  if (grp == 0) slope(xi);
  if (grp == (SPLIT ? 1 : 0) && t < TR) slope(-1);
  __syncthreads();
  double F[5];
  if (grp == 0) {
    const int lR = (xi + 2) * TR + r, lL = lR - TR, sR = (xi + 1) * TR + r, sL = sR - TR;
    auto ql = [&](int n) { return sq[n][lL]; };
    auto dql = [&](int n) { return sd[n][sL]; };
    auto qr = [&](int n) { return sq[n][lR]; };
    auto dqr = [&](int n) { return sd[n][sR]; };
    muscl_face<0>(ql, dql, qr, dqr, sq[QT][lL], c, F);
#pragma unroll
    for (int n = 0; n < 5; ++n) sF[n][t] = F[n];
  }
  __syncthreads();
  if (grp != 0 || xi >= W.nx) return;
  const Fab O = outf[W.box];
  if (!SPLIT && use_s1)
#pragma unroll
    for (int n = 0; n < 5; ++n) s1[n] = s1f[W.box](i, j, k, n);
#pragma unroll
  for (int n = 0; n < 5; ++n) {
    const double L = (bx.dxi[0] * (F[n] - sF[n][t + TR]) + (SPLIT ? st[n][t] : ty[n])) + (SPLIT ? st[5 + n][t] : tz[n]);
    tube_store(sa, sc, W.box, O, i, j, k, n, L, use_s1 ? s1[n] : 0.0, u[n], u[URHO], u[UMX]);
  }
}

}  // namespace

hipError_t launch_tube(int flux_euler, const TubeWork& tw, const BoxDev* boxes, const Closures& c, const StageArgs& sa,
                       const Fab* sin, const Fab* s1, const Fab* out, const XSide* xs, hipStream_t st) {
  if (tw.n <= 0) return hipSuccess;
  const dim3 g(unsigned(tw.n));
  constexpr int NX = TUBE_NX;
  static_assert(SX == TUBE_SPLIT_NX, "split bricks");
  if (flux_euler == 2) {
    if (tw.split)
      hipLaunchKernelGGL(k_weno_tube_split, g, dim3(15 * 64), 0, st, tw.d, boxes, c, sa, sin, s1, out, xs);
    else
      hipLaunchKernelGGL(k_weno_tube<NX>, g, dim3((NX + 1) * TR), 0, st, tw.d, boxes, c, sa, sin, s1, out, xs);
  } else if (flux_euler == 0) {
    if (tw.split)
      hipLaunchKernelGGL((k_muscl_tube<SX, true>), g, dim3((SX + 1) * TR * 3), 0, st, tw.d, boxes, c, sa, sin, s1, out,
                         xs);
    else
      hipLaunchKernelGGL((k_muscl_tube<NX, false>), g, dim3((NX + 1) * TR), 0, st, tw.d, boxes, c, sa, sin, s1, out,
                         xs);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace amr
