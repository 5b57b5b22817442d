// Fused KEEP (order 6) + viscous RHS and SSPRK stage update on tiles of 16x16
// columns that march in z; the operations of k_fused and their roundings.
//
// What bounded the form that orders 2 and 4 also take (k_fused, TGV 128^3, 212
// us a stage): six pairs evaluated for every x and y face and the own column's
// planes converted twice, in one workgroup a CU of one wave per SIMD.  Here
//   * a cell evaluates its three pairs A = (i, i-1), P = (i, i-2) and
//     Q = (i, i-3) per direction once; a face adds A, P of two and Q of three
//     cells (CentralKEEP.h:58-142, in that order).  x: lanes of a DPP row; y:
//     LDS; z: running sums of the two open faces in registers;
//   * the pairs of the cells 16 .. 18 past the tile that its faces read are
//     six sets of 32, one per half wave of waves 0 .. 2; wave 3 has the
//     ring's viscous fluxes;
//   * one plane of primitives in LDS, the plane above in registers, two
//     barriers a plane; a cell's x/y part waits two planes in registers for
//     its upper z face.
// Measured (MI355X, us a stage, k_fused -> this): TGV 128^3, tiles of 32 planes
// 212 -> 169; 96x80x72 one array per box, 16 planes 122 -> 99; 40x47x33, 1
// plane 41.8 -> 34.3.  What bounds it: 318 registers, one wave per SIMD, whose
// FP64 operations take 2/3 of an iteration (4.8 us).  Held to 256 registers it
// spilled (87): two workgroups a CU, but 261 us.
#include "kernels.h"
#include "fused_common.h"
#include "tile16.h"

namespace amr {

namespace {

using namespace fusedk;
using tile16::dpp_row;
using tile16::NRING;
using tile16::NT;
using tile16::RB;
using tile16::ring_cell;
using tile16::TX;
using tile16::TY;
using tile16::uniform;

constexpr int HX = 3, RX = TX + 2 * HX, RY = TY + 2 * HX, PL = RX * RY;
constexpr int ROW_SHL1 = 0x101, ROW_SHL2 = 0x102, ROW_SHR1 = 0x111;
// pairs of the cells past the tile: A of cell 16, P of 16 and 17, Q of 16 .. 18
constexpr int NKIND = 6;
// published pairs: co0 A_y of row 16, co1 P_y of rows 0 .. 17, co2 Q_y of rows
// 0 .. 18, the x pairs of the cells past the tile; viscous fluxes: y of rows
// -1 .. 16, x of columns -1, 16 and 15
constexpr int E_P = TX, E_Q = E_P + (TY + 2) * TX, E_X = E_Q + (TY + 3) * TX, E_END = E_X + NKIND * TY;
constexpr int V_X = (TY + 2) * TX, V_END = V_X + 3 * TY;

// LDS cell of a thread's halo load: ring threads load their ring cell, threads
// 0 .. 131 the two cells beyond it on each side and the ring's corners (no
// other corner is read); -1 for threads with none.
__device__ __forceinline__ int halo_cell(int tid) {
  int i, j;
  if (tid >= RB) {
    bool isx;
    ring_cell(tid - RB, isx, i, j);
  } else if (tid < 128) {
    const int side = tid >> 5, s = tid & 15, far = (tid >> 4) & 1;
    const int d = side & 1 ? TX + 1 + far : -2 - far;
    i = side < 2 ? d : s;
    j = side < 2 ? s : d;
  } else if (tid < 132) {
    i = tid & 1 ? TX : -1;
    j = tid & 2 ? TY : -1;
  } else {
    return -1;
  }
  return (j + HX) * RX + i + HX;
}

struct Cell {
  double rho, u, v, w, T, p;
};
__device__ __forceinline__ Cell lds_cell(const double* sq, int idx) {
  return Cell{sq[QRHO * PL + idx], sq[QU * PL + idx], sq[QV * PL + idx],
              sq[QW * PL + idx],   sq[QT * PL + idx], sq[QPRES * PL + idx]};
}
template <int NRM>
__device__ __forceinline__ void pair_terms(const Cell& a, const Cell& b, double cv, double co, double t[5]) {
  keep_terms<NRM>(a.rho, a.u, a.v, a.w, cv * a.T, a.p, b.rho, b.u, b.v, b.w, cv * b.T, b.p, t);
#pragma unroll
  for (int n = 0; n < 5; ++n) t[n] = co * t[n];
}

template <bool LEVEL, bool UCS, bool SRC>
__global__ void __launch_bounds__(NT, 1)
k_fused_keep6(const TileDev* __restrict__ tiles, const BoxDev* __restrict__ boxes, Closures c, double co0, double co1,
              double co2, StageArgs sa, WrapArgs wa, Cover cov, UncovSrc us, const Fab* __restrict__ s1f,
              const Fab* __restrict__ sinf, const Fab* __restrict__ outf) {
  __shared__ double s_q[NPRIM * PL];             // primitives of the plane
  __shared__ double s_e[5][E_END];               // published pairs (one stride: constant LDS offsets)
  __shared__ double s_v[4][V_END];               // published viscous fluxes
  __shared__ double s_fy[5][TY * TX];            // y faces 1 .. 16
  __shared__ double s_fx[5][TY];                 // x faces 16
  __shared__ unsigned s_um[UCS ? 2 * NT : 1];

  const TileDev T = tiles[blockIdx.x];
  if (T.nz <= 0 || !box_active(sa, T.box)) return;  // uniform: the whole workgroup leaves
  const StageCoef sc0 = box_stage(sa, T.box);
  const int mode = __builtin_amdgcn_readfirstlane(sc0.mode);
  const double sca = uniform(sc0.a), scb = uniform(sc0.b), scc = uniform(sc0.c), scd = uniform(sc0.d);
  const double dxi0 = boxes[T.box].dxi[0], dxi1 = boxes[T.box].dxi[1], dxi2 = boxes[T.box].dxi[2];
  const Fab S = sinf[T.box];
  const Fab O = outf[T.box];
  const bool use_s1 = __builtin_amdgcn_readfirstlane(mode != 2 && sca != 0.0);
  const Fab S1 = use_s1 ? s1f[T.box] : S;
  const bool has_src = SRC && sa.src != nullptr;
  const Fab SR = has_src ? sa.src[T.box] : S;  // user_source FAB (valid cells)
  const int tid = threadIdx.x;
  const int ti = tid % TX, tj = tid / TX;
  const int gi = T.i0 + ti, gj = T.j0 + tj;
  const int xhi = LEVEL ? cov.hi[0] : boxes[T.box].hi[0], yhi = LEVEL ? cov.hi[1] : boxes[T.box].hi[1];
  const int xcap = xhi + NGHOST, ycap = yhi + NGHOST;
  const bool own_in = gi <= xhi && gj <= yhi;
  guint* cbits = (guint*)cov.bits;  // coverage bitmap (level tiles)
  const int cplane = cov.nb[0] * cov.nb[1];
  const int ccol = own_in ? max((gj - cov.lo[1]) >> cov.sh, 0) * cov.nb[0] + max((gi - cov.lo[0]) >> cov.sh, 0) : 0;
  const int k0 = T.k0, nz = T.nz;
  const double cv = c.cv;
  const int own = (tj + HX) * RX + (ti + HX);
  // (a-b)*0.5*dxinv is evaluated as (a-b)*(0.5*dxinv): exact in IEEE
  // arithmetic for normal numbers (scaling by 0.5 is exact)
  const double hx = uniform(0.5 * dxi0), hy = uniform(0.5 * dxi1), hz = uniform(0.5 * dxi2);

  const bool ring = tid >= RB;
  bool rx;
  int ra, rb;
  ring_cell(tid & 63, rx, ra, rb);
  const int ring_idx = (rb + HX) * RX + (ra + HX);
  const int rdst = rx ? V_X + (tid & 31) : (rb + 1) * TX + ra;
  // cell past the tile whose pair this thread (waves 0 .. 2) evaluates
  const int ekind = tid >> 5, es = tid & 15;
  const bool ex_ = (tid & 16) == 0;  // x (columns past the tile), else y
  const int edist = ekind == 0 ? 1 : (ekind < 3 ? 2 : 3), epos = TX + (ekind < 3 ? max(ekind - 1, 0) : ekind - 3);
  const int estr = ex_ ? 1 : RX;
  const int eidx = (ex_ ? es + HX : epos + HX) * RX + (ex_ ? epos + HX : es + HX);
  const int edst = ex_ ? E_X + ekind * TY + es : (ekind == 0 ? es : (ekind < 3 ? E_P : E_Q) + epos * TX + es);
  const double eco = ekind == 0 ? co0 : (ekind < 3 ? co1 : co2);

  // load slots: 0 the own cell, 1 the halo cell (lanes with none load their
  // own cell again)
  const int hcell = halo_cell(tid);
  auto load_cell = [&](int s) { return s == 0 || hcell < 0 ? own : hcell; };
  const gdouble* sbase = gptr(S.p) + S.off;
  int loff[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int cell = load_cell(s);
    int x = min(T.i0 - HX + cell % RX, xcap), y = min(T.j0 - HX + cell / RX, ycap);
    if (wa.on) {
      x = x < wa.lo[0] ? x + wa.len[0] : (x >= wa.lo[0] + wa.len[0] ? x - wa.len[0] : x);
      y = y < wa.lo[1] ? y + wa.len[1] : (y >= wa.lo[1] + wa.len[1] ? y - wa.len[1] : y);
    }
    loff[s] = x + y * int(S.js);
  }
  // ghost cells no box covers come from U^n (UCS): bit b of the lane's mask
  // for load slot s is set when the cell is such a ghost cell in plane block
  // zb0 + b; at most UNCOV_MAX_ZBLK blocks per tile
  const int zb0 = (k0 - HX - us.lo[2]) >> us.sh;
  const gdouble* u0base = sbase;
  if (UCS) {
    const Fab U0 = us.u0[T.box];
    u0base = gptr(U0.p) + U0.off;
    const int zb1 = (k0 + nz + 2 - us.lo[2]) >> us.sh;
    guint* ubits = (guint*)us.bits;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int cell = load_cell(s);
      const int bx = (min(T.i0 - HX + cell % RX, xcap) - us.lo[0]) >> us.sh;
      const int by = (min(T.j0 - HX + cell / RX, ycap) - us.lo[1]) >> us.sh;
      const bool inxy = bx >= 0 && bx < us.nb[0] && by >= 0 && by < us.nb[1];
      unsigned m = 0u;
      for (int zb = zb0; zb <= zb1; ++zb) {
        if (inxy && zb >= 0 && zb < us.nb[2]) {
          const int bit = (zb * us.nb[1] + by) * us.nb[0] + bx;
          if ((ubits[bit >> 5] >> (bit & 31)) & 1u) m |= 1u << (zb - zb0);
        }
      }
      s_um[s * NT + tid] = m;
    }
  }
  double pre[2][5];
  // `below`, `above`: may be a plane that the array holds in part (Cover)
  auto load = [&](int s, int p, bool below = false, bool above = false) {
    if (wa.on) p = p < wa.lo[2] ? p + wa.len[2] : (p >= wa.lo[2] + wa.len[2] ? p - wa.len[2] : p);
    const gdouble* pb = sbase + int64_t(p) * S.ks;
    int o = loff[s];
    if (LEVEL && below && p < cov.lo[2] - 2) o = max(o, cov.below);
    if (LEVEL && above && p > cov.hi[2] + 2) o = min(o, cov.above);
    if (UCS && ((s_um[s * NT + tid] >> (((p - us.lo[2]) >> us.sh) - zb0)) & 1u)) {
      const gdouble* pu = u0base + int64_t(p) * S.ks;
#pragma unroll
      for (int n = 0; n < 5; ++n) pre[s][n] = pu[n * S.ns + o];
    } else {
#pragma unroll
      for (int n = 0; n < 5; ++n) pre[s][n] = pb[n * S.ns + o];
    }
  };
  // the finished plane's own conserved state and s1, clamped into the valid
  // region: overhanging lanes load there and never store
  const int soff = min(gi, xhi) + min(gj, yhi) * int(S.js);
  const gdouble* s1base = gptr(S1.p) + S1.off;
  const int s1off = min(gi, xhi) + min(gj, yhi) * int(S1.js);
  double sv[5], s1v[5];
  auto load_epilogue = [&](int p) {
    const gdouble* pb = sbase + int64_t(p) * S.ks;
#pragma unroll
    for (int n = 0; n < 5; ++n) sv[n] = pb[n * S.ns + soff];
    if (use_s1) {
      const gdouble* p1 = s1base + int64_t(p) * S1.ks;
#pragma unroll
      for (int n = 0; n < 5; ++n) s1v[n] = p1[n * S1.ns + s1off];
    }
  };

  // own column: planes p, p-2, p-3 (p-1 is in LDS); halo cell of plane p
  double q0[NPRIM], q2[NPRIM], q3[NPRIM], hn[NPRIM];
  double rm1[4] = {0, 0, 0, 0};  // u, v, w, T of the ring cell, plane p-2
  auto convert = [&](int s, double q[NPRIM]) {
    cons2prim(pre[s][0], pre[s][1], pre[s][2], pre[s][3], pre[s][4], c, q);
  };
  auto store_plane = [&]() {
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) s_q[n * PL + own] = q0[n];
    if (hcell >= 0)
#pragma unroll
      for (int n = 0; n < NPRIM; ++n) s_q[n * PL + hcell] = hn[n];
  };

  load(0, k0 - 3, true);
  convert(0, q3);
  load(0, k0 - 2);
  load(1, k0 - 2);
  convert(0, q2);
  convert(1, hn);
#pragma unroll
  for (int n = 0; n < 4; ++n) rm1[n] = hn[QU + n];
  load(0, k0 - 1);
  load(1, k0 - 1);
  convert(0, q0);
  convert(1, hn);
  store_plane();
  load(0, k0);
  load(1, k0);
  __syncthreads();

  // z faces: fa the face p-2 up to its last term, fb the face p-1 up to P(p-1),
  // q1t = co2 Q(p-1), fz_prev the finished face p-3; viscous z flux of planes
  // p-3 and p-2; x/y parts of the planes p-3 and p-2
  double fa[5] = {0, 0, 0, 0, 0}, fb[5] = {0, 0, 0, 0, 0}, q1t[5] = {0, 0, 0, 0, 0}, fz_prev[5] = {0, 0, 0, 0, 0};
  double va[4] = {0, 0, 0, 0}, vb[4] = {0, 0, 0, 0};
  double xy3[5] = {0, 0, 0, 0, 0}, xy2[5] = {0, 0, 0, 0, 0};

  for (int p = k0; p <= k0 + nz + 2; ++p) {
    const bool inner = p > k0 && p <= k0 + nz;  // x/y work on the plane in LDS, p - 1
    // ---- own column of plane p: its z pairs
    convert(0, q0);
    if (p < k0 + nz + 2) load(0, p + 1, false, true);
    {
      const Cell o{q0[QRHO], q0[QU], q0[QV], q0[QW], q0[QT], q0[QPRES]};
      double t[5];
      pair_terms<2>(o, Cell{q3[QRHO], q3[QU], q3[QV], q3[QW], q3[QT], q3[QPRES]}, cv, co2, t);
      if (p >= k0 + 2) {
        double fz[5];
#pragma unroll
        for (int n = 0; n < 5; ++n) fz[n] = fa[n] + t[n];
#pragma unroll
        for (int n = 0; n < 4; ++n) fz[n + 1] = __builtin_fma(0.5, va[n] + vb[n], fz[n + 1]);
        const int kp = p - 3;
        if (kp >= k0) {
          bool write = own_in;
          if (LEVEL) {
            const int bit = ((kp - cov.lo[2]) >> cov.sh) * cplane + ccol;
            write = write && ((cbits[bit >> 5] >> (bit & 31)) & 1u);
          }
          if (write) {
            gdouble* po = gptr(O.p) + O.idx(gi, gj, kp);
            double L[5];
#pragma unroll
            for (int n = 0; n < 5; ++n) {
              L[n] = xy3[n] + dxi2 * (fz_prev[n] - fz[n]);
              if (has_src) L[n] = L[n] + SR(gi, gj, kp, n);  // user_source
            }
            if (SRC && sa.bfx != 0.0) {  // body-force user_source (exm/Channel/prob.h:189-193)
              L[UMX] = L[UMX] + sv[URHO] * sa.bfx;
              L[UET] = L[UET] + sv[UMX] * sa.bfx;
            }
            // stage_combine, its choices (uniform) taken once for the five
            if (use_s1) {
              if (mode == 0)
#pragma unroll
                for (int n = 0; n < 5; ++n) po[n * O.ns] = sca * s1v[n] + scb * (scc * sv[n] + scd * L[n]);
              else
#pragma unroll
                for (int n = 0; n < 5; ++n) po[n * O.ns] = (sca * s1v[n] + scc * sv[n]) + scd * L[n];
            } else if (mode == 2) {
#pragma unroll
              for (int n = 0; n < 5; ++n) po[n * O.ns] = L[n];
            } else {
#pragma unroll
              for (int n = 0; n < 5; ++n) {
                const double v = scc * sv[n] + scd * L[n];
                po[n * O.ns] = mode == 0 ? scb * v : v;
              }
            }
          }
        }
#pragma unroll
        for (int n = 0; n < 5; ++n) fz_prev[n] = fz[n];
      }
      if (p == k0 + nz + 2) break;  // uniform: that was the tile's last face
      double s[5];
      pair_terms<2>(o, Cell{q2[QRHO], q2[QU], q2[QV], q2[QW], q2[QT], q2[QPRES]}, cv, co1, s);
#pragma unroll
      for (int n = 0; n < 5; ++n) {
        fa[n] = ((fb[n] + s[n]) + q1t[n]) + t[n];
        fb[n] = s[n];
        q1t[n] = t[n];
      }
      pair_terms<2>(o, lds_cell(s_q, own), cv, co0, s);
#pragma unroll
      for (int n = 0; n < 5; ++n) fb[n] = s[n] + fb[n];
    }
    convert(1, hn);
    if (p < k0 + nz) load(1, p + 1);
    // ---- plane p-1: viscous fluxes
    double vx[4];
    {
      VDer d;
      d.ux = s_q[QU * PL + own];
      d.uy = s_q[QV * PL + own];
      d.uz = s_q[QW * PL + own];
      d.T = s_q[QT * PL + own];
      const int e = own + 1, w = own - 1, nn = own + RX, s = own - RX;
      d.dudx = (s_q[QU * PL + e] - s_q[QU * PL + w]) * hx;
      d.dvdx = (s_q[QV * PL + e] - s_q[QV * PL + w]) * hx;
      d.dwdx = (s_q[QW * PL + e] - s_q[QW * PL + w]) * hx;
      d.dTdx = (s_q[QT * PL + e] - s_q[QT * PL + w]) * hx;
      d.dudy = (s_q[QU * PL + nn] - s_q[QU * PL + s]) * hy;
      d.dvdy = (s_q[QV * PL + nn] - s_q[QV * PL + s]) * hy;
      d.dwdy = (s_q[QW * PL + nn] - s_q[QW * PL + s]) * hy;
      d.dTdy = (s_q[QT * PL + nn] - s_q[QT * PL + s]) * hy;
      d.dudz = (q0[QU] - q2[QU]) * hz;
      d.dvdz = (q0[QV] - q2[QV]) * hz;
      d.dwdz = (q0[QW] - q2[QW]) * hz;
      d.dTdz = (q0[QT] - q2[QT]) * hz;
      double vz[4], vy[4];
      if (inner) {
        visc_flux<true, true, true>(d, c, vx, vy, vz);
#pragma unroll
        for (int n = 0; n < 4; ++n) s_v[n][tid + TX] = vy[n];
        if (ti == TX - 1)
#pragma unroll
          for (int n = 0; n < 4; ++n) s_v[n][V_X + 2 * TY + tj] = vx[n];
      } else {
        visc_flux<false, false, true>(d, c, vx, vy, vz);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        va[n] = vb[n];
        vb[n] = vz[n];
      }
    }
    // ---- plane p-1: pairs of the own cell in x and y
    double fx[5], px[5], qx[5], ay[5];
    if (inner) {
      const Cell o = lds_cell(s_q, own);
      double t[5];
      pair_terms<1>(o, lds_cell(s_q, own - RX), cv, co0, ay);
      pair_terms<1>(o, lds_cell(s_q, own - 2 * RX), cv, co1, t);
#pragma unroll
      for (int n = 0; n < 5; ++n) s_e[n][E_P + tid] = t[n];
      pair_terms<1>(o, lds_cell(s_q, own - 3 * RX), cv, co2, t);
#pragma unroll
      for (int n = 0; n < 5; ++n) s_e[n][E_Q + tid] = t[n];
      pair_terms<0>(o, lds_cell(s_q, own - 1), cv, co0, fx);
      pair_terms<0>(o, lds_cell(s_q, own - 2), cv, co1, px);
#pragma unroll
      for (int n = 0; n < 5; ++n) fx[n] += px[n];
      pair_terms<0>(o, lds_cell(s_q, own - 3), cv, co2, qx);
      if (!ring) {
        // pairs of the cells past the tile
        const Cell a = lds_cell(s_q, eidx), b = lds_cell(s_q, eidx - edist * estr);
        keep_terms_xy(ex_, a.rho, a.u, a.v, a.w, cv * a.T, a.p, b.rho, b.u, b.v, b.w, cv * b.T, b.p, t);
#pragma unroll
        for (int n = 0; n < 5; ++n) s_e[n][edst] = eco * t[n];
      }
    }
    if (ring) {
      double rs[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) rs[n] = s_q[(QU + n) * PL + ring_idx];
      if (inner) {
        VDer g;
        const int r = ring_idx;
        g.ux = rs[0];
        g.uy = rs[1];
        g.uz = rs[2];
        g.T = rs[3];
        const int e = r + 1, w = r - 1, nn = r + RX, s = r - RX;
        g.dudx = (s_q[QU * PL + e] - s_q[QU * PL + w]) * hx;
        g.dvdx = (s_q[QV * PL + e] - s_q[QV * PL + w]) * hx;
        g.dwdx = (s_q[QW * PL + e] - s_q[QW * PL + w]) * hx;
        g.dTdx = (s_q[QT * PL + e] - s_q[QT * PL + w]) * hx;
        g.dudy = (s_q[QU * PL + nn] - s_q[QU * PL + s]) * hy;
        g.dvdy = (s_q[QV * PL + nn] - s_q[QV * PL + s]) * hy;
        g.dwdy = (s_q[QW * PL + nn] - s_q[QW * PL + s]) * hy;
        g.dTdy = (s_q[QT * PL + nn] - s_q[QT * PL + s]) * hy;
        g.dudz = (hn[QU] - rm1[0]) * hz;
        g.dvdz = (hn[QV] - rm1[1]) * hz;
        g.dwdz = (hn[QW] - rm1[2]) * hz;
        g.dTdz = (hn[QT] - rm1[3]) * hz;
        double gx[4], gy[4], gz[4];
        visc_flux<true, true, false>(g, c, gx, gy, gz);
#pragma unroll
        for (int n = 0; n < 4; ++n) s_v[n][rdst] = rx ? gx[n] : gy[n];
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) rm1[n] = rs[n];
    }
    double q1[NPRIM];
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) q1[n] = s_q[n * PL + own];
    __syncthreads();  // the plane's readers are done, its pairs and fluxes visible
    store_plane();
    // ---- faces of plane p-1
    double fy[5];
    if (inner) {
#pragma unroll
      for (int n = 0; n < 5; ++n) {
        const double* sp = s_e[n] + tid;
        const double* sx = s_e[n] + E_X + tj;
        fx[n] += dpp_row<ROW_SHL1>(sx[1 * TY], px[n]);
        fx[n] += qx[n];
        fx[n] += dpp_row<ROW_SHL1>(sx[3 * TY], qx[n]);
        fx[n] += dpp_row<ROW_SHL2>(ti == TX - 1 ? sx[4 * TY] : sx[3 * TY], qx[n]);
        fy[n] = ((((ay[n] + sp[E_P]) + sp[E_P + TX]) + sp[E_Q]) + sp[E_Q + TX]) + sp[E_Q + 2 * TX];
        if (n > 0) {
          fx[n] = __builtin_fma(0.5, dpp_row<ROW_SHR1>(s_v[n - 1][V_X + tj], vx[n - 1]) + vx[n - 1], fx[n]);
          fy[n] = __builtin_fma(0.5, s_v[n - 1][tid] + s_v[n - 1][tid + TX], fy[n]);
        }
        if (tj > 0) s_fy[n][tid - TX] = fy[n];
      }
      if (tid < 2 * TX) {
        // faces 16
        const bool isx = tid < TY;
        const int e1 = isx ? E_X + TY + es : E_P + TY * TX + es, d1 = isx ? TY : TX;
        const int e3 = isx ? E_X + 3 * TY + es : E_Q + TY * TX + es;
#pragma unroll
        for (int n = 0; n < 5; ++n) {
          const double* se = s_e[n];
          double f = ((((se[isx ? E_X + es : es] + se[e1]) + se[e1 + d1]) + se[e3]) + se[e3 + d1]) + se[e3 + 2 * d1];
          if (n > 0) {
            const double* v = s_v[n - 1];
            f = __builtin_fma(0.5, isx ? v[V_X + 2 * TY + es] + v[V_X + TY + es] : v[TY * TX + es] + v[(TY + 1) * TX + es], f);
          }
          (isx ? s_fx[n] : s_fy[n] + (TY - 1) * TX)[es] = f;
        }
      }
    }
    if (p >= k0 + 2) load_epilogue(p - 2);  // for the next plane's first section
    __syncthreads();  // faces and plane p visible
#pragma unroll
    for (int n = 0; n < 5; ++n) {
      xy3[n] = xy2[n];
      if (inner) {
        const double fxr = dpp_row<ROW_SHL1>(s_fx[n][tj], fx[n]);
        xy2[n] = dxi0 * (fx[n] - fxr) + dxi1 * (fy[n] - s_fy[n][tid]);
      }
    }
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) {
      q3[n] = q2[n];
      q2[n] = q1[n];
    }
  }
}

template <bool SRC>
void launch(const TileDev* tiles, int ntiles, const BoxDev* boxes, const Closures& c, const double co[3],
            const StageArgs& sa, const WrapArgs& wa, const Cover& cov, const UncovSrc& us, const Fab* s1,
            const Fab* sin, const Fab* out, hipStream_t st) {
#define AMR_KEEP6(LEVEL_, UCS_)                                                                                      \
  hipLaunchKernelGGL((k_fused_keep6<LEVEL_, UCS_, SRC>), dim3(ntiles), dim3(NT), 0, st, tiles, boxes, c, co[0], co[1], \
                     co[2], sa, wa, cov, us, s1, sin, out)
  if (cov.on && us.on) AMR_KEEP6(true, true);
  else if (cov.on) AMR_KEEP6(true, false);
  else if (us.on) AMR_KEEP6(false, true);
  else AMR_KEEP6(false, false);
#undef AMR_KEEP6
}

}  // namespace

hipError_t launch_fused_keep6(const TileDev* tiles, int ntiles, const BoxDev* boxes, const Closures& c,
                              const double co[3], const StageArgs& sa, const WrapArgs& wa, const Cover& cov,
                              const UncovSrc& us, const Fab* s1, const Fab* sin, const Fab* out, hipStream_t st) {
  if (sa.src != nullptr || sa.bfx != 0.0) launch<true>(tiles, ntiles, boxes, c, co, sa, wa, cov, us, s1, sin, out, st);
  else launch<false>(tiles, ntiles, boxes, c, co, sa, wa, cov, us, s1, sin, out, st);
  return hipGetLastError();
}

}  // namespace amr
