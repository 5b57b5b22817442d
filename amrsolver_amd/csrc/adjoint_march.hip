// Reverse mode of a whole stage of a periodic level held as one array (KEEP
// order 2/4, with or without the viscous terms): the transposes of the KEEP
// pairs, of the viscous cell fluxes, of cons2prim and of the stage combination
// in one kernel, cells as in the pass-structured reverse (k_adj_visc,
// k_adj_cell), of src/rhs/CNS_hydro_K.h:15-34,108-172,254-261,
// src/rhs/CentralKEEP.h:40-145 and src/tim/CNS_advance.cpp:375-391.
//
// What bounded the passes (128x64x64, 98 us a stage): 190 gathered values a
// cell through L1, and 36 values a cell (primitives, adjoints of the viscous
// differences) written by one pass and read by the next.  Here a workgroup of
// 16x16 cells marches in z:
//   * the plane's primitives and stage adjoints, halo 2, lie in LDS; state and
//     adjoint of the next plane are loaded during the plane's work;
//   * z: each pair is transposed once, into running sums of both its planes
//     (three planes of sums, values and adjoints in registers), and so is a
//     cell's viscous z flux into the planes above and below;
//   * x and y: a cell gathers its pairs from the LDS plane; the adjoints of the
//     viscous differences go to the neighbours by DPP (x: a tile row is one DPP
//     row of 16 lanes) and LDS (y).  The cells of the ring around the tile,
//     whose differences reach into it, belong to the last wave.
// Measured (MI355X, 128x64x64 KEEP4 viscous, tiles of 4 planes): 98 -> 44 us a
// reverse stage alone, the checkpointed run of 20 steps 8.28 -> 5.51 ms.  What
// bounds it now: FP64 chains at two waves per SIMD (235 VGPRs), and at 4 planes
// a tile two iterations in six are pipeline.
#include "kernels.h"
#include "fused_common.h"
#include "tile16.h"

// no bits are pinned to another kernel here: products and sums contract
#pragma clang fp contract(fast)
#include "adjoint_point.h"

namespace amr {

namespace {

using namespace fusedk;
using namespace tile16;

constexpr int OB = RB - NOUT;  // first thread of the halo cells that are not ring cells

// The adjoint weights of the viscous cell fluxes (a, b, c: half the central
// differences of the stage adjoint in x, y, z, components 1..4) turned into
// the adjoints of the stresses.
struct StressAdj {
  double gxx, gxy, gxz, gyy, gyz, gzz, s3;
};
__device__ __forceinline__ StressAdj stress_adj(const double a[5], const double b[5], const double cc[5], double ux,
                                                double uy, double uz) {
  StressAdj r;
  r.gxx = -a[UMX] - a[UET] * ux;
  r.gxy = -a[UMY] - a[UET] * uy - b[UMX] - b[UET] * ux;
  r.gxz = -a[UMZ] - a[UET] * uz - cc[UMX] - cc[UET] * ux;
  r.gyy = -b[UMY] - b[UET] * uy;
  r.gyz = -b[UMZ] - b[UET] * uz - cc[UMY] - cc[UET] * uy;
  r.gzz = -cc[UMZ] - cc[UET] * uz;
  r.s3 = (r.gxx + r.gyy + r.gzz) * (1.0 / 3.0);
  return r;
}
// adjoints of the u, v, w, T differences in direction D (h = 1/(2 dx))
template <int D>
__device__ __forceinline__ void diff_adj(const StressAdj& s, double mu, double kk, double aE, double h, double e[4]) {
  const double hm = h * mu;
  e[0] = D == 0 ? 2.0 * hm * (s.gxx - s.s3) : hm * (D == 1 ? s.gxy : s.gxz);
  e[1] = D == 1 ? 2.0 * hm * (s.gyy - s.s3) : hm * (D == 0 ? s.gxy : s.gyz);
  e[2] = D == 2 ? 2.0 * hm * (s.gzz - s.s3) : hm * (D == 0 ? s.gxz : s.gyz);
  e[3] = -h * kk * aE;
}

constexpr int per_cu(int h, bool visc) { return h == 1 && !visc ? 3 : 2; }

// Reverse of the stage on the workgroup's tile.  mode 0: lam_sin (=|+=)
// b (c lam_out + d G), mode 1: c lam_out + d G, mode 2: G; lam_s1 (+=|=)
// a lam_out (s1_mode 1|2, 0 none), G = (d dSdt / d S)^T lam_out.
template <int H, bool VISC>
__global__ void __launch_bounds__(NT, per_cu(H, VISC))
k_adj_march(const TileDev* __restrict__ tiles, const BoxDev* __restrict__ boxes, Closures c, double co0, double co1,
            StageCoef sc, WrapArgs wa, const Fab* __restrict__ sinf, const Fab* __restrict__ lamf, const Fab* lam_s1,
            const Fab* lam_sin, int accumulate, int s1_mode) {
  __shared__ double s_q[NPRIM * PL];  // primitives of the plane
  __shared__ double s_l[NCONS * PL];  // stage adjoint of the plane
  __shared__ double s_y[4][(TY + 2) * TX];  // adjoints of y differences, rows -1 .. 16
  __shared__ double s_x[4][2 * TY];         // of x differences, columns -1 and 16
  __shared__ double s_r[NCONS][NRING];      // ring cells' stage adjoint, plane below

  const TileDev T = tiles[blockIdx.x];
  if (T.nz <= 0) return;  // uniform: the whole workgroup leaves
  const int tid = threadIdx.x, ti = tid % TX, tj = tid / TX;
  const int gi = T.i0 + ti, gj = T.j0 + tj;
  const int xhi = boxes[T.box].hi[0], yhi = boxes[T.box].hi[1];
  const bool own_in = gi <= xhi && gj <= yhi;
  const double dxi0 = boxes[T.box].dxi[0], dxi1 = boxes[T.box].dxi[1], dxi2 = boxes[T.box].dxi[2];
  const double hx = uniform(0.5 * dxi0), hy = uniform(0.5 * dxi1), hz = uniform(0.5 * dxi2);
  const Fab S = sinf[T.box], L = lamf[T.box], Li = lam_sin[T.box];
  const Fab L1 = s1_mode ? lam_s1[T.box] : Li;
  const int k0 = T.k0, nz = T.nz;
  const double cv = c.cv;
  const int own = (tj + HX) * RX + (ti + HX);
  const int hcell = halo_cell<OB>(tid);
  const bool ring = tid >= RB;
  bool rx;
  int ra, rb;
  ring_cell(tid & 63, rx, ra, rb);
  const int ring_idx = (rb + HX) * RX + (ra + HX);

  // offsets of the own and the halo column in both arrays; columns past the
  // box's halo load its last one, and images wrap
  int so[2], lo[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int cell = s == 0 || hcell < 0 ? own : hcell;
    int x = min(T.i0 - HX + cell % RX, xhi + HX), y = min(T.j0 - HX + cell / RX, yhi + HX);
    x = x < wa.lo[0] ? x + wa.len[0] : (x >= wa.lo[0] + wa.len[0] ? x - wa.len[0] : x);
    y = y < wa.lo[1] ? y + wa.len[1] : (y >= wa.lo[1] + wa.len[1] ? y - wa.len[1] : y);
    so[s] = x + y * int(S.js);
    lo[s] = x + y * int(L.js);
  }
  const gdouble* sbase = gptr(S.p) + S.off;
  const gdouble* lbase = gptr(L.p) + L.off;
  double pu[2][NCONS], pl[2][NCONS];  // state and adjoint: own column of the next plane, halo column of this one
  auto load = [&](int s, int p) {
    p = p < wa.lo[2] ? p + wa.len[2] : (p >= wa.lo[2] + wa.len[2] ? p - wa.len[2] : p);
    const gdouble* pb = sbase + int64_t(p) * S.ks;
    const gdouble* qb = lbase + int64_t(p) * L.ks;
#pragma unroll
    for (int n = 0; n < NCONS; ++n) pu[s][n] = pb[n * S.ns + so[s]];
#pragma unroll
    for (int n = 0; n < NCONS; ++n) pl[s][n] = qb[n * L.ns + lo[s]];
  };

  // own column: primitives and stage adjoint of planes p and p-2 (plane p-1 is
  // in LDS) and the sums of the adjoint of the primitives of the three
  double q0[NPRIM], q2[NPRIM], l0[NCONS], l2[NCONS], g0[NPRIM], g1[NPRIM], g2[NPRIM];
#pragma unroll
  for (int n = 0; n < NPRIM; ++n) g1[n] = g2[n] = 0.0;

  // the plane whose own column is in q0, l0 and whose halo column is loaded
  auto store_plane = [&]() {
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) s_q[n * PL + own] = q0[n];
#pragma unroll
    for (int n = 0; n < NCONS; ++n) s_l[n * PL + own] = l0[n];
    if (hcell >= 0) {
      double hq[NPRIM];
      cons2prim(pu[1][0], pu[1][1], pu[1][2], pu[1][3], pu[1][4], c, hq);
#pragma unroll
      for (int n = 0; n < NPRIM; ++n) s_q[n * PL + hcell] = hq[n];
#pragma unroll
      for (int n = 0; n < NCONS; ++n) s_l[n * PL + hcell] = pl[1][n];
    }
  };
  auto own_column = [&](double q[NPRIM], double l[NCONS]) {
    cons2prim(pu[0][0], pu[0][1], pu[0][2], pu[0][3], pu[0][4], c, q);
#pragma unroll
    for (int n = 0; n < NCONS; ++n) l[n] = pl[0][n];
  };

  // plane k0-2 (own column) and k0-1
  load(0, k0 - 2);
  load(1, k0 - 1);
  own_column(q2, l2);
  section();
  load(0, k0 - 1);
  section();
  own_column(q0, l0);
  store_plane();
  section();
  load(0, k0);
  __syncthreads();
  for (int p = k0; p <= k0 + nz + 1; ++p) {
    const bool inner = p > k0 && p <= k0 + nz;  // k = p - 1, the plane in LDS, is the tile's
    // ---- own column of plane p and its z pairs
    own_column(q0, l0);
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) g0[n] = 0.0;
    {
      double w[NCONS];
      if (p <= k0 + nz) {
        double q1[NPRIM];
#pragma unroll
        for (int n = 0; n < NPRIM; ++n) q1[n] = s_q[n * PL + own];
#pragma unroll
        for (int n = 0; n < NCONS; ++n) w[n] = co0 * dxi2 * (l0[n] - s_l[n * PL + own]);
        keep_pair_vjp<2, true, true>(w, q0, q1, cv, g0, g1);
      }
      section();
      if (H == 2) {
#pragma unroll
        for (int n = 0; n < NCONS; ++n) w[n] = co1 * dxi2 * (l0[n] - l2[n]);
        keep_pair_vjp<2, true, true>(w, q0, q2, cv, g0, g2);
      }
    }
    section();
    // ---- plane k: viscous terms
    double ex[4] = {0.0, 0.0, 0.0, 0.0};
    // behind a uniform branch (wa.on is always set here): without one the order 4
    // kernel takes 256 registers and spills seven, with it 235
    if (VISC && wa.on) {
      double a[NCONS], b[NCONS], cc[NCONS];
#pragma unroll
      for (int n = 1; n < NCONS; ++n) {
        a[n] = hx * (s_l[n * PL + own + 1] - s_l[n * PL + own - 1]);
        b[n] = hy * (s_l[n * PL + own + RX] - s_l[n * PL + own - RX]);
        cc[n] = hz * (l0[n] - l2[n]);
      }
      const double T1 = s_q[QT * PL + own];
      const StressAdj sa = stress_adj(a, b, cc, s_q[QU * PL + own], s_q[QV * PL + own], s_q[QW * PL + own]);
      section();
      const double mu = visc(c, T1), kk = cond(c, T1, mu);
      section();
      double e[4];
      diff_adj<2>(sa, mu, kk, cc[UET], hz, e);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        g0[QU + n] += e[n];
        g2[QU + n] -= e[n];
      }
      if (inner) {
        diff_adj<0>(sa, mu, kk, a[UET], hx, ex);
        diff_adj<1>(sa, mu, kk, b[UET], hy, e);
#pragma unroll
        for (int n = 0; n < 4; ++n) s_y[n][(tj + 1) * TX + ti] = e[n];
        section();
        // the cell's own values: u, v, w through the work of the stresses,
        // T through mu and k
        double dx[4], dy[4], dz[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const double* f = s_q + (QU + n) * PL;
          dx[n] = hx * (f[own + 1] - f[own - 1]);
          dy[n] = hy * (f[own + RX] - f[own - RX]);
          dz[n] = hz * (q0[QU + n] - q2[QU + n]);
        }
        const double third = (dx[0] + dy[1] + dz[2]) * (1.0 / 3.0);
        const double sxx = 2.0 * (dx[0] - third), syy = 2.0 * (dy[1] - third), szz = 2.0 * (dz[2] - third);
        const double sxy = dy[0] + dx[1], sxz = dz[0] + dx[2], syz = dz[1] + dy[2];
        const double am = mu * a[UET], bm = mu * b[UET], cm = mu * cc[UET];
        g1[QU] -= am * sxx + bm * sxy + cm * sxz;
        g1[QV] -= am * sxy + bm * syy + cm * syz;
        g1[QW] -= am * sxz + bm * syz + cm * szz;
        const double gmu = sa.gxx * sxx + sa.gyy * syy + sa.gzz * szz + sa.gxy * sxy + sa.gxz * sxz + sa.gyz * syz;
        const double gk = a[UET] * dx[3] + b[UET] * dy[3] + cc[UET] * dz[3];
        section();
        double dmu, dk;
        transport_derivs(c, T1, mu, kk, dmu, dk);
        g1[QT] += gmu * dmu - gk * dk;
      }
    }
    section();
    // ---- plane p-2 is complete: cons2prim and the stage combination
    // transposed (T = p/(rho R), p = (gamma-1)(E - |m|^2/(2 rho)), v = m/rho)
    const int ko = p - 2;
    if (ko >= k0 && own_in) {
      const double rinv = 1.0 / q2[QRHO];
      const double ux = q2[QU], uy = q2[QV], uz = q2[QW];
      const double gp = g2[QPRES] + g2[QT] * rinv / c.Rspec;
      const double gr = g2[QRHO] - g2[QT] * q2[QT] * rinv;
      const double gg = c.gm1 * gp;
      double G[NCONS];
      G[URHO] = gr + 0.5 * (ux * ux + uy * uy + uz * uz) * gg - (g2[QU] * ux + g2[QV] * uy + g2[QW] * uz) * rinv;
      G[UMX] = g2[QU] * rinv - ux * gg;
      G[UMY] = g2[QV] * rinv - uy * gg;
      G[UMZ] = g2[QW] * rinv - uz * gg;
      G[UET] = gg;
      gdouble* po = gptr(Li.p) + Li.idx(gi, gj, ko);
      gdouble* p1 = gptr(L1.p) + L1.idx(gi, gj, ko);
      const double a = sc.mode == 2 ? 0.0 : sc.a;
      // lam_s1 may be lam_sin: its old value is then what lam_sin gets here
      const bool same = s1_mode != 0 && p1 == po;
#pragma unroll
      for (int n = 0; n < NCONS; ++n) {
        double v = G[n];
        if (sc.mode == 0) v = sc.b * (sc.c * l2[n] + sc.d * v);
        else if (sc.mode == 1) v = sc.c * l2[n] + sc.d * v;
        if (accumulate) v = po[n * Li.ns] + v;
        if (same) v = s1_mode == 2 ? a * l2[n] : v + a * l2[n];
        po[n * Li.ns] = v;
      }
      if (s1_mode != 0 && !same && (s1_mode == 2 || a != 0.0)) {
#pragma unroll
        for (int n = 0; n < NCONS; ++n) p1[n * L1.ns] = s1_mode == 2 ? a * l2[n] : p1[n * L1.ns] + a * l2[n];
      }
    }
    section();
    if (p == k0 + nz + 1) break;  // uniform: that was the last plane of the tile
    load(1, p);
    load(0, p + 1);
    section();
    // ---- plane k: x and y pairs
    double q1[NPRIM], l1[NCONS];
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) q1[n] = s_q[n * PL + own];
#pragma unroll
    for (int n = 0; n < NCONS; ++n) l1[n] = s_l[n * PL + own];
    if (inner) {
#pragma unroll
      for (int l = 1; l <= H; ++l) {
        const double cl = l == 1 ? co0 : co1;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const int st = d == 0 ? 1 : RX;
          const double cw = cl * (d == 0 ? dxi0 : dxi1);
#pragma unroll
          for (int side = 0; side < 2; ++side) {
            const int nb = side == 0 ? own - l * st : own + l * st;
            double w[NCONS], qn[NPRIM];
#pragma unroll
            for (int n = 0; n < NCONS; ++n) {
              const double ln = s_l[n * PL + nb];
              w[n] = side == 0 ? cw * (l1[n] - ln) : cw * (ln - l1[n]);
            }
#pragma unroll
            for (int n = 0; n < NPRIM; ++n) qn[n] = s_q[n * PL + nb];
            if (d == 0) keep_pair_vjp<0, true, false>(w, q1, qn, cv, g1, nullptr);
            else keep_pair_vjp<1, true, false>(w, q1, qn, cv, g1, nullptr);
            section();
          }
        }
      }
    }
    section();
    // ---- plane k: adjoints of the ring cells' differences
    if (VISC && inner && ring) {
      double e[4], ra_[NCONS], rb_[NCONS], rc_[NCONS];
#pragma unroll
      for (int n = 1; n < NCONS; ++n) {
        ra_[n] = hx * (s_l[n * PL + ring_idx + 1] - s_l[n * PL + ring_idx - 1]);
        rb_[n] = hy * (s_l[n * PL + ring_idx + RX] - s_l[n * PL + ring_idx - RX]);
        rc_[n] = hz * (pl[1][n] - s_r[n][tid - RB]);
      }
      const StressAdj rs = stress_adj(ra_, rb_, rc_, s_q[QU * PL + ring_idx], s_q[QV * PL + ring_idx],
                                      s_q[QW * PL + ring_idx]);
      const double rT = s_q[QT * PL + ring_idx];
      const double rmu = visc(c, rT), rkk = cond(c, rT, rmu);
      if (rx) {
        diff_adj<0>(rs, rmu, rkk, ra_[UET], hx, e);
#pragma unroll
        for (int n = 0; n < 4; ++n) s_x[n][tid & 31] = e[n];
      } else {
        diff_adj<1>(rs, rmu, rkk, rb_[UET], hy, e);
#pragma unroll
        for (int n = 0; n < 4; ++n) s_y[n][(rb + 1) * TX + ra] = e[n];
      }
    }
    if (VISC && ring)
#pragma unroll
      for (int n = 1; n < NCONS; ++n) s_r[n][tid - RB] = s_l[n * PL + ring_idx];
    __syncthreads();  // plane k has been read, the differences' adjoints are there
    store_plane();
    if (VISC && inner) {
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const double xl = dpp_row<ROW_SHR1>(s_x[n][tj], ex[n]);
        const double xr = dpp_row<ROW_SHL1>(s_x[n][TY + tj], ex[n]);
        g1[QU + n] += (xl - xr) + (s_y[n][tj * TX + ti] - s_y[n][(tj + 2) * TX + ti]);
      }
    }
    // ---- next plane
#pragma unroll
    for (int n = 0; n < NPRIM; ++n) {
      q2[n] = q1[n];
      g2[n] = g1[n];
      g1[n] = g0[n];
    }
#pragma unroll
    for (int n = 0; n < NCONS; ++n) l2[n] = l1[n];
    __syncthreads();  // plane p stands
  }
}

}  // namespace

bool adj_march_supported(const amr_scheme_t& s) {
  return s.rhs_euler && s.flux_euler == 1 && !s.art_diss && (s.order_keep == 2 || s.order_keep == 4);
}

int adj_march_per_cu(const amr_scheme_t& s) { return per_cu(s.order_keep / 2, s.rhs_visc != 0); }

hipError_t launch_adj_march(const amr_scheme_t& s, const TileDev* tiles, int ntiles, const BoxDev* boxes,
                            const Closures& c, const StageCoef& sc, const WrapArgs& wa, const Fab* sin,
                            const Fab* lam_out, const Fab* lam_s1, const Fab* lam_sin, bool accumulate, int s1_mode,
                            hipStream_t st) {
  if (!adj_march_supported(s) || !wa.on) return hipErrorInvalidValue;
  if (ntiles == 0) return hipSuccess;
  double co[3] = {0.0, 0.0, 0.0};
  keep_coefficients(s.order_keep, co);
#define AMR_MARCH(HH, VV)                                                                                           \
  hipLaunchKernelGGL((k_adj_march<HH, VV>), dim3(unsigned(ntiles)), dim3(NT), 0, st, tiles, boxes, c, co[0], co[1], sc, \
                     wa, sin, lam_out, lam_s1, lam_sin, accumulate ? 1 : 0, lam_s1 ? s1_mode : 0)
  if (s.order_keep == 4) {
    if (s.rhs_visc) AMR_MARCH(2, true);
    else AMR_MARCH(2, false);
  } else {
    if (s.rhs_visc) AMR_MARCH(1, true);
    else AMR_MARCH(1, false);
  }
#undef AMR_MARCH
  return hipGetLastError();
}

}  // namespace amr
