// Fused KEEP (order 2/4) + viscous RHS and SSPRK stage update, the
// self-loading form: 16x16 columns marched in z like k_fused, rearranged so
// that each KEEP pair and each neighbour cell is used once.
//
// What bounded the first form (TGV 256^3, 766 us a stage): VALU issue and LDS
// each about half busy at two waves per SIMD.  A face of order 4 needs the
// pairs (i, i-1), (i, i-2) and (i+1, i-1); the last one is the next face's
// (i, i-2), and the cells i-1 and i+1 are also the ones the viscous
// derivatives read.  So here every thread
//   1. reads its cell's four x/y neighbours from LDS once, computes its
//      viscous cell fluxes and per direction the pairs A = (i, i-1) and
//      P = (i+1, i-1), and publishes co1 P and the viscous flux of y (LDS);
//   2. forms the x face below its cell from its left neighbour's P and
//      viscous flux (DPP row shifts: a tile row is one DPP row of 16 lanes),
//      the y face from the row below, publishes the y face, and forms the z
//      face and the epilogue of the plane below from its own column;
//   3. takes the next faces (DPP, LDS) and the plane's x/y differences.
// Two barriers per plane; the next plane is converted straight from the
// prefetch registers (no thread reads a cell of it that it did not load) and
// stored once the plane's readers are done, so LDS holds one plane.  The own
// column's conserved state is kept in LDS until its epilogue two planes on
// (the first form reads it from L2 again).  Wave 3 computes the ring cells'
// viscous fluxes, wave 0 their pairs and the faces at i = 16 and j = 16; the
// roles rotate over the SIMDs from workgroup to workgroup.  The published
// values share one LDS stride per array, so that their addresses are
// immediate offsets: with strides per lane the kernel spilled, and every
// reload waited for the prefetch (835 us instead of 675).
//
// Measured (MI355X, us a stage; first form and its earlier self-loading
// variant with three and two barriers and 6 pairs per x/y face pair -> this):
// TGV 256^3 KEEP4 766 -> 660, KEEP2 640 -> 586; 192x160x128 with one array
// per box 216 -> 189; the channel 96x128x64 between bc 6 walls, fills
// included, 222 (pass-structured kernels) -> 65.  What bounds it now: latency
// at two waves per SIMD (243 VGPRs, 78 KB of LDS); the VALU is busy about
// half of the time, the LDS a fifth.
#include "kernels.h"
#include "fused_common.h"
#include "tile16.h"

namespace amr {

namespace {

using namespace fusedk;
using namespace tile16;

constexpr int OB = 64;                      // first thread of those
constexpr int NEDGE = 2 * TY + TX;          // x faces 16, y faces 16, x faces 0: formed by threads 0 .. 47
constexpr int E_XLO = (TY + 1) * TX, E_HI = E_XLO + 2 * TY, E_END = E_HI + NEDGE;
constexpr int F_X = TY * TX, F_END = F_X + 2 * TY;

struct Cell {
  double rho, u, v, w, T, p;
};
__device__ __forceinline__ Cell lds_cell(const double* sq, int idx) {
  return Cell{sq[QRHO * PL + idx], sq[QU * PL + idx], sq[QV * PL + idx],
              sq[QW * PL + idx],   sq[QT * PL + idx], sq[QPRES * PL + idx]};
}
template <int NRM>
__device__ __forceinline__ void pair_terms(const Cell& a, const Cell& b, double cv, double t[5]) {
  keep_terms<NRM>(a.rho, a.u, a.v, a.w, cv * a.T, a.p, b.rho, b.u, b.v, b.w, cv * b.T, b.p, t);
}
__device__ __forceinline__ void pair_terms_xy(bool isx, const Cell& a, const Cell& b, double cv, double t[5]) {
  keep_terms_xy(isx, a.rho, a.u, a.v, a.w, cv * a.T, a.p, b.rho, b.u, b.v, b.w, cv * b.T, b.p, t);
}

// WALL: tables with bc 6 walls in y: the y faces next to a wall take order 2
// (k_keep_wall's rule: faces lo .. lo+H-1 of a box at the lower wall,
// hi-H+1 .. hi at the upper), the cell fluxes of the ghost row outside it
// one-sided y derivatives (k_visc_wall's).  UCS, SRC, NB as in k_fused.
template <int H, bool LEVEL, bool UCS, bool SRC, int NB, bool WALL>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
k_fused_self(const TileDev* __restrict__ tiles, const BoxDev* __restrict__ boxes, Closures c, double co0, double co1,
             StageArgs sa, WrapArgs wa, Cover cov, UncovSrc us, NbMap nbm, WallRows wr, const Fab* __restrict__ s1f,
             const Fab* __restrict__ sinf, const Fab* __restrict__ outf) {
  static_assert(H == 1 || H == 2, "KEEP order 2 or 4");
  static_assert(!(NB && (UCS || LEVEL)) && !(WALL && (NB || UCS || LEVEL)), "unsupported combination");
  constexpr int NP = H == 2 ? 5 : 0;  // published pair terms
  constexpr int NE = NP + 4;          // published values per cell: co1 P, viscous flux
  __shared__ double s_q[NPRIM * PL];       // primitives of the plane
  // co1 P and viscous flux that cells publish: y of rows -1 .. 15; x of the
  // cells below the x faces 16 and 0 (i = 15, -1); the cells above the faces
  // i = 16, j = 16 and i = 0 (one stride for all: constant LDS offsets)
  __shared__ double s_e[NE][E_END];
  __shared__ double s_a[5][NEDGE];         // co0 A of the cells above those faces
  __shared__ double s_f[5][F_END];         // y faces 1 .. 16, x faces 16, x faces 0
  __shared__ double s_u[2][NCONS][NT];     // own column's conserved state, two planes
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
  // the wave roles (ring fluxes on wave 3, ring pairs on wave 0) rotate so
  // that the two workgroups of a CU load its SIMDs differently
  const int tid = (threadIdx.x + 64 * ((blockIdx.x >> 3) + (blockIdx.x >> 8))) & (NT - 1);
  const int ti = tid % TX, tj = tid / TX;
  const int gi = T.i0 + ti, gj = T.j0 + tj;
  const int xhi = LEVEL ? cov.hi[0] : boxes[T.box].hi[0], yhi = LEVEL ? cov.hi[1] : boxes[T.box].hi[1];
  const int xcap = xhi + NGHOST, ycap = yhi + NGHOST;
  const bool own_in = gi <= xhi && gj <= yhi;
  // coverage bitmap (level tiles; tiles per box write every cell of the box)
  guint* cbits = (guint*)cov.bits;
  const int cplane = cov.nb[0] * cov.nb[1];
  const int ccol = own_in ? max((gj - cov.lo[1]) >> cov.sh, 0) * cov.nb[0] + max((gi - cov.lo[0]) >> cov.sh, 0) : 0;
  const int k0 = T.k0, nz = T.nz;
  const double cv = c.cv;
  const int own = (tj + HX) * RX + (ti + HX);
  // (a-b)*0.5*dxinv is evaluated as (a-b)*(0.5*dxinv): exact in IEEE
  // arithmetic for normal numbers (scaling by 0.5 is exact)
  const double hx = uniform(0.5 * dxi0), hy = uniform(0.5 * dxi1), hz = uniform(0.5 * dxi2);
  // next to bc 6 walls: y faces of order 2 (j <= wlo, or whi <= j <= wtop)
  // and ghost rows with one-sided derivatives
  int wlo = INT_MIN, whi = INT_MAX, wtop = INT_MIN, grow_lo = INT_MIN, grow_hi = INT_MIN;
  if (WALL) {
    const int blo = boxes[T.box].lo[1], bhi = boxes[T.box].hi[1];
    if (wr.lo_wall && blo == wr.dlo) {
      if (H == 2) wlo = blo + H - 1;
      grow_lo = blo - 1;
    }
    if (wr.hi_wall && bhi == wr.dhi) {
      if (H == 2) {
        whi = bhi - H + 1;
        wtop = bhi;
      }
      grow_hi = bhi + 1;
    }
  }

  const bool ring = tid >= RB;
  bool rx;  // ring cell of threads RB.. (viscous flux) and 0..63 (pairs)
  int ra, rb;
  ring_cell(tid & 63, rx, ra, rb);
  const int ring_idx = (rb + HX) * RX + (ra + HX);
  const int rstride = rx ? 1 : RX;
  // where they publish: right and top cells are the upper cells of the edge
  // faces, the left ones the lower cells of face 0, the bottom ones row -1
  const bool rhi = (tid & 16) != 0;
  const int rslot = (rx ? 0 : TY) + (tid & 15);
  const int rp = rhi ? E_HI + rslot : (rx ? E_XLO + TY + (tid & 15) : (tid & 15));

  // load slots: 0 the own cell, 1 the halo cell (lanes with none load their
  // own cell again)
  const int hcell = halo_cell<OB>(tid);
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
  // NB: per slot the element offset of its column in the array that holds it
  // and, for NB 1, that array's plane and component strides; refreshed when
  // the plane enters another block of the owner map (uniform over the tile)
  constexpr int NBS = NB == 1 ? 2 : 1;
  int nks[NBS], nns[NBS];
  int nzb = INT_MIN;
  auto nb_refresh = [&](int p) {
    const int zb = (p - nbm.dlo[2]) >> nbm.sh;
    if (zb == nzb) return;
    nzb = zb;
    int pw = p, zbw = zb;
    if (nbm.per[2]) {
      pw = p < nbm.dlo[2] ? p + nbm.len[2] : (p >= nbm.dlo[2] + nbm.len[2] ? p - nbm.len[2] : p);
      zbw = (pw - nbm.dlo[2]) >> nbm.sh;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int cell = load_cell(s);
      const int x = min(T.i0 - HX + cell % RX, xcap), y = min(T.j0 - HX + cell / RX, ycap);
      int xw = x, yw = y;
      if (nbm.per[0]) xw = x < nbm.dlo[0] ? x + nbm.len[0] : (x >= nbm.dlo[0] + nbm.len[0] ? x - nbm.len[0] : x);
      if (nbm.per[1]) yw = y < nbm.dlo[1] ? y + nbm.len[1] : (y >= nbm.dlo[1] + nbm.len[1] ? y - nbm.len[1] : y);
      const int ob = nbm.owner[(int64_t(zbw) * nbm.nb[1] + ((yw - nbm.dlo[1]) >> nbm.sh)) * nbm.nb[0] +
                               ((xw - nbm.dlo[0]) >> nbm.sh)];
      if (ob >= 0) {
        const Fab F = sinf[ob];
        loff[s] = int((F.p - S.p) + (F.off - S.off) + xw + int64_t(yw) * F.js + int64_t(pw - p) * F.ks);
        if constexpr (NB == 1) {
          nks[s] = int(F.ks);
          nns[s] = int(F.ns);
        }
      } else {
        loff[s] = x + y * int(S.js);
        if constexpr (NB == 1) {
          nks[s] = int(S.ks);
          nns[s] = int(S.ns);
        }
      }
    }
  };
  // ghost cells no box covers come from U^n (UCS): bit b of the lane's mask
  // for load slot s is set when the cell is such a ghost cell in plane block
  // zb0 + b; at most UNCOV_MAX_ZBLK blocks per tile
  const int zb0 = (k0 - HX - us.lo[2]) >> us.sh;
  const gdouble* u0base = sbase;
  if (UCS) {
    const Fab U0 = us.u0[T.box];
    u0base = gptr(U0.p) + U0.off;
    const int zb1 = (k0 + nz + 1 - us.lo[2]) >> us.sh;
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
  auto load_plane = [&](int p, int s_first = 0, int s_last = 1) {
    if constexpr (NB == 1) {
      if (s_last == 1) nb_refresh(p);
#pragma unroll
      for (int s = s_first; s <= s_last; ++s) {
        const int o = loff[s] + p * nks[s];
#pragma unroll
        for (int n = 0; n < 5; ++n) pre[s][n] = sbase[int64_t(o) + n * nns[s]];
      }
      return;
    }
    if constexpr (NB == 2) if (s_last == 1) nb_refresh(p);  // then the plain form with the refreshed offsets
    if (!NB && wa.on) p = p < wa.lo[2] ? p + wa.len[2] : (p >= wa.lo[2] + wa.len[2] ? p - wa.len[2] : p);
    const gdouble* pb = sbase + int64_t(p) * S.ks;
    if (UCS) {
      const int b = ((p - us.lo[2]) >> us.sh) - zb0;
      const gdouble* pu = u0base + int64_t(p) * S.ks;
#pragma unroll
      for (int s = s_first; s <= s_last; ++s) {
        if ((s_um[s * NT + tid] >> b) & 1u) {
#pragma unroll
          for (int n = 0; n < 5; ++n) pre[s][n] = pu[n * S.ns + loff[s]];
        } else {
#pragma unroll
          for (int n = 0; n < 5; ++n) pre[s][n] = pb[n * S.ns + loff[s]];
        }
      }
    } else {
#pragma unroll
      for (int s = s_first; s <= s_last; ++s)
#pragma unroll
        for (int n = 0; n < 5; ++n) pre[s][n] = pb[n * S.ns + loff[s]];
    }
  };
  const gdouble* s1base = gptr(S1.p) + S1.off;
  const int s1off = min(gi, xhi) + min(gj, yhi) * int(S1.js);  // overhanging lanes load there and never store

  double qm1[NPRIM], qs[NPRIM], qn[NPRIM], hn[NPRIM];
  double rm1[4];  // u, v, w, T of the ring cell, plane below
  auto convert = [&]() {
    cons2prim(pre[0][0], pre[0][1], pre[0][2], pre[0][3], pre[0][4], c, qn);
    if (hcell >= 0) cons2prim(pre[1][0], pre[1][1], pre[1][2], pre[1][3], pre[1][4], c, hn);
  };
  auto store_plane = [&]() {
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) s_q[n * PL + own] = qn[n];
    if (hcell >= 0)
#pragma unroll
      for (int n = 0; n < NPRIM; ++n) s_q[n * PL + hcell] = hn[n];
  };
  auto keep_u = [&](int p) {
#pragma unroll
    for (int n = 0; n < NCONS; ++n) s_u[p & 1][n][tid] = pre[0][n];
  };

  // planes k0-2 (own and ring column only) and k0-1
  load_plane(k0 - 2);
  convert();
#pragma unroll
  for (int n = 0; n < NPRIM; ++n) qm1[n] = qn[n];
#pragma unroll
  for (int n = 0; n < 4; ++n) rm1[n] = hn[QU + n];
  load_plane(k0 - 1);
  convert();
  keep_u(k0 - 1);
  store_plane();
#pragma unroll
  for (int n = 0; n < NPRIM; ++n) qs[n] = qn[n];
  load_plane(k0);
  __syncthreads();

  double pfz_prev[4] = {0, 0, 0, 0}, pfz_cur[4];
  double fz_prev[5] = {0, 0, 0, 0, 0};
  double zcarry[5] = {0, 0, 0, 0, 0};  // z pair (c+1, c-1) terms for the next plane
  double xy_prev[5] = {0, 0, 0, 0, 0};

  // where the thread publishes co1 P_y and its viscous y flux (the row below
  // is TX before), and lanes 0 (upper cell of face 0) and 15 (lower cell of
  // face 16) their co1 P_x and viscous x flux
  const int pe = (tj + 1) * TX + ti;
  const int xp = ti == 0 ? E_HI + TX + TY + tj : E_XLO + tj;
  // lower cell and result slot of the edge face of threads 0 .. 47
  const int elo = tid < TY ? E_XLO + tid : (tid < TY + TX ? TY * TX + tid - TY : E_XLO + tid - TX);
  const int edst = tid < TY ? F_X + tid : (tid < TY + TX ? (TY - 1) * TX + tid - TY : F_X + tid - TX);
  // next to a wall the y face is the pair alone, coefficient 1
  const bool two = WALL && (gj <= wlo || (gj >= whi && gj <= wtop));
  const bool two16 = WALL && (T.j0 + TY <= wlo || (T.j0 + TY >= whi && T.j0 + TY <= wtop));
  double s1v[5];
  auto load_s1 = [&](int p) {
    const gdouble* p1 = s1base + int64_t(p) * S1.ks;
#pragma unroll
    for (int n = 0; n < 5; ++n) s1v[n] = p1[n * S1.ns + s1off];
  };

  for (int cpl = k0 - 1; cpl <= k0 + nz; ++cpl) {
    const bool inner = cpl >= k0 && cpl < k0 + nz;  // x/y work on this plane
    // ---- phase 1
    convert();
    load_plane(min(cpl + 2, k0 + nz + 1), 1, 1);
    double vx[4];
    {
      VDer d;
      d.ux = qs[QU];
      d.uy = qs[QV];
      d.uz = qs[QW];
      d.T = qs[QT];
      const int e = own + 1, w = own - 1, nn = own + RX, s = own - RX;
      d.dudx = (s_q[QU * PL + e] - s_q[QU * PL + w]) * hx;
      d.dvdx = (s_q[QV * PL + e] - s_q[QV * PL + w]) * hx;
      d.dwdx = (s_q[QW * PL + e] - s_q[QW * PL + w]) * hx;
      d.dTdx = (s_q[QT * PL + e] - s_q[QT * PL + w]) * hx;
      d.dudy = (s_q[QU * PL + nn] - s_q[QU * PL + s]) * hy;
      d.dvdy = (s_q[QV * PL + nn] - s_q[QV * PL + s]) * hy;
      d.dwdy = (s_q[QW * PL + nn] - s_q[QW * PL + s]) * hy;
      d.dTdy = (s_q[QT * PL + nn] - s_q[QT * PL + s]) * hy;
      if (WALL && gj == grow_hi) {  // an overhanging row just outside the upper wall
        const int s2 = own - 2 * RX;
        d.dudy = (3 * qs[QU] - 4 * s_q[QU * PL + s] + s_q[QU * PL + s2]) * hy;
        d.dvdy = (3 * qs[QV] - 4 * s_q[QV * PL + s] + s_q[QV * PL + s2]) * hy;
        d.dwdy = (3 * qs[QW] - 4 * s_q[QW * PL + s] + s_q[QW * PL + s2]) * hy;
        d.dTdy = (3 * qs[QT] - 4 * s_q[QT * PL + s] + s_q[QT * PL + s2]) * hy;
      }
      d.dudz = (qn[QU] - qm1[QU]) * hz;
      d.dvdz = (qn[QV] - qm1[QV]) * hz;
      d.dwdz = (qn[QW] - qm1[QW]) * hz;
      d.dTdz = (qn[QT] - qm1[QT]) * hz;
      double vy[4];
      if (inner) {
        visc_flux<true, true, true>(d, c, vx, vy, pfz_cur);
#pragma unroll
        for (int n = 0; n < 4; ++n) s_e[NP + n][pe] = vy[n];
      } else {
        visc_flux<false, false, true>(d, c, vx, vy, pfz_cur);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (cpl >= k0) {
      // z face at cpl - 1/2 from the own column (planes c-1, c, c+1)
      double fz[5], t[5];
      zterms(qs, qm1, cv, t);  // (c, c-1)
#pragma unroll
      for (int n = 0; n < 5; ++n) fz[n] = co0 * t[n];
      if (H == 2) {
        // (c, c-2) is the previous plane's (c+1, c-1), carried in registers
        keep_accum(co1, zcarry, fz);
        zterms(qn, qm1, cv, zcarry);  // (c+1, c-1)
        keep_accum(co1, zcarry, fz);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) fz[n + 1] = __builtin_fma(0.5, pfz_prev[n] + pfz_cur[n], fz[n + 1]);
      if (cpl > k0) {
        // the plane below is complete
        const int kp = cpl - 1;
        bool write = own_in;
        if (LEVEL) {
          const int bit = ((kp - cov.lo[2]) >> cov.sh) * cplane + ccol;
          write = write && ((cbits[bit >> 5] >> (bit & 31)) & 1u);
        }
        if (write) {
          gdouble* po = gptr(O.p) + O.idx(gi, gj, kp);
          double sv[5], L[5];
#pragma unroll
          for (int n = 0; n < 5; ++n) {
            sv[n] = s_u[kp & 1][n][tid];
            L[n] = xy_prev[n] + dxi2 * (fz_prev[n] - fz[n]);
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
    } else if (H == 2) {
      zterms(qn, qm1, cv, zcarry);  // (k0, k0-2) for the first face
    }
    if (cpl == k0 + nz) break;  // uniform: the last plane has no x/y work
    // the plane above replaces the finished one; the prefetch of the next
    // takes the registers it leaves
    keep_u(cpl + 1);
    load_plane(min(cpl + 2, k0 + nz + 1), 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    double fx[5], ay[5];
    if (inner) {
      const Cell o{qs[QRHO], qs[QU], qs[QV], qs[QW], qs[QT], qs[QPRES]};
      double t[5];
      {
        const Cell e = lds_cell(s_q, own + 1), w = lds_cell(s_q, own - 1);
        pair_terms<0>(o, w, cv, t);
#pragma unroll
        for (int n = 0; n < 5; ++n) fx[n] = co0 * t[n];
        if (ti == 0)
#pragma unroll
          for (int n = 0; n < 5; ++n) s_a[n][TX + TY + tj] = fx[n];
        if (H == 2) {
          pair_terms<0>(e, w, cv, t);
#pragma unroll
          for (int n = 0; n < 5; ++n) {
            t[n] = co1 * t[n];
            fx[n] += dpp_row<ROW_SHR1>(0.0, t[n]);
            fx[n] += t[n];
          }
          if (ti == 0 || ti == TX - 1)
#pragma unroll
            for (int n = 0; n < 5; ++n) s_e[n][xp] = t[n];
        }
        if (ti == 0 || ti == TX - 1)
#pragma unroll
          for (int n = 0; n < 4; ++n) s_e[NP + n][xp] = vx[n];
#pragma unroll
        for (int n = 0; n < 4; ++n) fx[n + 1] = __builtin_fma(0.5, dpp_row<ROW_SHR1>(0.0, vx[n]) + vx[n], fx[n + 1]);
      }
      {
        const Cell nn = lds_cell(s_q, own + RX), s = lds_cell(s_q, own - RX);
        pair_terms<1>(o, s, cv, t);
#pragma unroll
        for (int n = 0; n < 5; ++n) ay[n] = (two ? 1.0 : co0) * t[n];
        if (H == 2) {
          pair_terms<1>(nn, s, cv, t);
#pragma unroll
          for (int n = 0; n < 5; ++n) s_e[n][pe] = co1 * t[n];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (inner && tid < NRING) {
      // pairs of the ring cells (left and bottom cells: P only)
      const Cell a = lds_cell(s_q, ring_idx + rstride), b = lds_cell(s_q, ring_idx - rstride);
      double t[5];
      if (H == 2) {
        pair_terms_xy(rx, a, b, cv, t);
#pragma unroll
        for (int n = 0; n < 5; ++n) s_e[n][rp] = co1 * t[n];
      }
      if (rhi) {
        const Cell q = lds_cell(s_q, ring_idx);
        const double ca = two16 && !rx ? 1.0 : co0;
        pair_terms_xy(rx, q, b, cv, t);
#pragma unroll
        for (int n = 0; n < 5; ++n) s_a[n][rslot] = ca * t[n];
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
        if (WALL && !rx) {
          const int row = T.j0 + rb;
          if (row == grow_lo) {
            const int n1 = r + RX, n2 = r + 2 * RX;
            g.dudy = (-s_q[QU * PL + n2] + 4 * s_q[QU * PL + n1] - 3 * rs[0]) * hy;
            g.dvdy = (-s_q[QV * PL + n2] + 4 * s_q[QV * PL + n1] - 3 * rs[1]) * hy;
            g.dwdy = (-s_q[QW * PL + n2] + 4 * s_q[QW * PL + n1] - 3 * rs[2]) * hy;
            g.dTdy = (-s_q[QT * PL + n2] + 4 * s_q[QT * PL + n1] - 3 * rs[3]) * hy;
          } else if (row == grow_hi) {
            const int n1 = r - RX, n2 = r - 2 * RX;
            g.dudy = (3 * rs[0] - 4 * s_q[QU * PL + n1] + s_q[QU * PL + n2]) * hy;
            g.dvdy = (3 * rs[1] - 4 * s_q[QV * PL + n1] + s_q[QV * PL + n2]) * hy;
            g.dwdy = (3 * rs[2] - 4 * s_q[QW * PL + n1] + s_q[QW * PL + n2]) * hy;
            g.dTdy = (3 * rs[3] - 4 * s_q[QT * PL + n1] + s_q[QT * PL + n2]) * hy;
          }
        }
        g.dudz = (hn[QU] - rm1[0]) * hz;
        g.dvdz = (hn[QV] - rm1[1]) * hz;
        g.dwdz = (hn[QW] - rm1[2]) * hz;
        g.dTdz = (hn[QT] - rm1[3]) * hz;
        double gx[4], gy[4], gz[4];
        visc_flux<true, true, false>(g, c, gx, gy, gz);
#pragma unroll
        for (int n = 0; n < 4; ++n) s_e[NP + n][rp] = rx ? gx[n] : gy[n];
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) rm1[n] = rs[n];
    }
    // ---- phase 2: the plane's readers are done, its pairs and fluxes visible
    __syncthreads();
    store_plane();
    if (use_s1 && inner) load_s1(cpl);  // for the next iteration's epilogue
    double fy[5];
    if (inner) {
#pragma unroll
      for (int n = 0; n < 5; ++n) {
        fy[n] = ay[n];
        if (H == 2) {
          double f = ay[n] + s_e[n][pe - TX];
          f += s_e[n][pe];
          fy[n] = two ? fy[n] : f;
        }
        if (n > 0) fy[n] = __builtin_fma(0.5, s_e[NP + n - 1][pe - TX] + s_e[NP + n - 1][pe], fy[n]);
      }
      if (tj > 0)
#pragma unroll
        for (int n = 0; n < 5; ++n) s_f[n][(tj - 1) * TX + ti] = fy[n];
      if (tid < NEDGE) {
        const bool isy = tid >= TY && tid < TY + TX;
#pragma unroll
        for (int n = 0; n < 5; ++n) {
          double f = s_a[n][tid];
          if (H == 2) {
            double g = f + s_e[n][elo];
            g += s_e[n][E_HI + tid];
            f = two16 && isy ? f : g;
          }
          if (n > 0) f = __builtin_fma(0.5, s_e[NP + n - 1][elo] + s_e[NP + n - 1][E_HI + tid], f);
          s_f[n][edst] = f;
        }
      }
    }
    __syncthreads();  // faces and the next plane visible
    // ---- phase 3: the plane's x/y differences
    if (inner) {
#pragma unroll
      for (int n = 0; n < 5; ++n) {
        const double fxr = dpp_row<ROW_SHL1>(s_f[n][F_X + tj], fx[n]);
        const double fxl = ti == 0 ? s_f[n][F_X + TY + tj] : fx[n];
        xy_prev[n] = dxi0 * (fxl - fxr) + dxi1 * (fy[n] - s_f[n][tj * TX + ti]);
      }
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) pfz_prev[n] = pfz_cur[n];
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) {
      qm1[n] = qs[n];
      qs[n] = qn[n];
    }
  }
}

#define AMR_SELF_LAUNCH(LEVEL_, UCS_, SRC_, NB_, WALL_)                                                       \
  hipLaunchKernelGGL((k_fused_self<H, LEVEL_, UCS_, SRC_, NB_, WALL_>), dim3(ntiles), dim3(NT), 0, st, tiles, \
                     boxes, c, co[0], co[1], sa, wa, cov, us, nbm, wr, s1, sin, out)

template <int H, bool SRC>
void launch_h(const TileDev* tiles, int ntiles, const BoxDev* boxes, const Closures& c, const double co[3],
              const StageArgs& sa, const WrapArgs& wa, const Cover& cov, const UncovSrc& us, const NbMap& nbm,
              const WallRows& wr, const Fab* s1, const Fab* sin, const Fab* out, hipStream_t st) {
  if (wr.on) AMR_SELF_LAUNCH(false, false, SRC, 0, true);
  else if (nbm.on && nbm.ustride) AMR_SELF_LAUNCH(false, false, SRC, 2, false);
  else if (nbm.on) AMR_SELF_LAUNCH(false, false, SRC, 1, false);
  else if (cov.on && us.on) AMR_SELF_LAUNCH(true, true, SRC, 0, false);
  else if (cov.on) AMR_SELF_LAUNCH(true, false, SRC, 0, false);
  else if (us.on) AMR_SELF_LAUNCH(false, true, SRC, 0, false);
  else AMR_SELF_LAUNCH(false, false, SRC, 0, false);
}
#undef AMR_SELF_LAUNCH

}  // namespace

bool fused_self_supported(const amr_scheme_t& s, int tx, int ty) {
  return fused_supported(s, tx, ty) && s.order_keep <= 4 && s.rhs_visc && tx == TX && ty == TY;
}

hipError_t launch_fused_self(const amr_scheme_t& s, const FusedConfig& cfg, const WrapArgs& wa, const Cover& cov,
                             const UncovSrc& us, const TileDev* tiles, int ntiles, const BoxDev* boxes,
                             const Closures& c, const StageArgs& sa, const Fab* s1, const Fab* sin, const Fab* out,
                             hipStream_t st, const NbMap& nbm, const WallRows& wr) {
  if (!fused_self_supported(s, cfg.tx, cfg.ty) || (nbm.on && us.on) ||
      (wr.on && (nbm.on || us.on || cov.on)))
    return hipErrorInvalidValue;
  double co[3];
  keep_coefficients(s.order_keep, co);
  const bool src = sa.src != nullptr || sa.bfx != 0.0;
  auto launch = s.order_keep == 4 ? (src ? launch_h<2, true> : launch_h<2, false>)
                                  : (src ? launch_h<1, true> : launch_h<1, false>);
  launch(tiles, ntiles, boxes, c, co, sa, wa, cov, us, nbm, wr, s1, sin, out, st);
  return hipGetLastError();
}

}  // namespace amr
