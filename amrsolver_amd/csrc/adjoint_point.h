// Transposes of the point functions that the reverse kernels share (local to
// each file: one contracts their products and sums).
#pragma once

#include "cns_point.h"

namespace amr {
namespace {

// d mu / dT and d k / dT of the closures (Sutherland: mu (1.5/T - 1/(S+T)))
__device__ __forceinline__ void transport_derivs(const Closures& c, double T, double mu, double k, double& dmu,
                                                 double& dk) {
  dmu = c.visc_law == 0 ? 0.0 : mu * (1.5 / T - 1.0 / (c.Tvisc_ref + T));
  if (c.cond_law == 0) dk = 0.0;
  else if (c.cond_law == 1) dk = k * (1.5 / T - 1.0 / (c.Tcond_ref + T));
  else dk = dmu * c.cp / c.Pr;
}

// Reverse of one KEEP pair in direction NRM (keep_pair): w[5] is the weight
// of the pair's five flux components; adds (dP/dq1)^T w to g1 (G1) and
// (dP/dq2)^T w to g2 (G2), q = (rho, u, v, w, T, p), ie = cv T.
// With A = (rho1+rho2)(un1+un2) the pair is
//   P.w = A Gs + 0.5 (p1+p2) w[1+NRM] + 0.5 w[4] (p1 un2 + p2 un1),
//   Gs = w0/4 + sum_t w[1+t] (ut1+ut2)/8 + w[4] (ke/4 + (ie1+ie2)/8).
template <int NRM, bool G1, bool G2>
__device__ __forceinline__ void keep_pair_vjp(const double w[5], const double q1[6], const double q2[6], double cv,
                                              double g1[6], double g2[6]) {
  const double R = q1[QRHO] + q2[QRHO];
  const double un1 = q1[QU + NRM], un2 = q2[QU + NRM];
  const double U = un1 + un2;
  const double A = R * U;
  const double ke = 0.5 * (q1[QU] * q2[QU] + q1[QV] * q2[QV] + q1[QW] * q2[QW]);
  const double we = w[UET];
  double Gs = 0.25 * w[URHO] + we * (0.25 * ke + 0.125 * cv * (q1[QT] + q2[QT]));
#pragma unroll
  for (int t = 0; t < 3; ++t) Gs += 0.125 * w[UMX + t] * (q1[QU + t] + q2[QU + t]);
  const double A8 = 0.125 * A;
  if (G1) {
    g1[QRHO] += U * Gs;
#pragma unroll
    for (int t = 0; t < 3; ++t) g1[QU + t] += A8 * (w[UMX + t] + we * q2[QU + t]);
    g1[QU + NRM] += R * Gs + 0.5 * we * q2[QPRES];
    g1[QT] += A8 * we * cv;
    g1[QPRES] += 0.5 * (w[UMX + NRM] + we * un2);
  }
  if (G2) {
    g2[QRHO] += U * Gs;
#pragma unroll
    for (int t = 0; t < 3; ++t) g2[QU + t] += A8 * (w[UMX + t] + we * q1[QU + t]);
    g2[QU + NRM] += R * Gs + 0.5 * we * q1[QPRES];
    g2[QT] += A8 * we * cv;
    g2[QPRES] += 0.5 * (w[UMX + NRM] + we * un1);
  }
}

}  // namespace
}  // namespace amr
