// Device code of the short-range contact force, shared by the contact source
// and the tiled passes.
#pragma once

#include "pdg_internal.hpp"

namespace pdg {
namespace dev {

// One pair of the short-range force model seen from `cur` (position X,
// velocity V, volume vc) with neighbour `nb` (y, v, vn); returns false beyond
// the contact radius. fc: the force density on cur; fn (BOTH only): on nb.
// Expressions in the reference's order.
template <bool BOTH>
__device__ __forceinline__ bool contact_pair(const PairParams& P, const double X[3],
                                             const double V[3], double vc, const double y[3],
                                             const double v[3], double vn, double fc[3],
                                             double fn[3]) {
  const double d0 = y[0] - X[0], d1 = y[1] - X[1], d2 = y[2] - X[2];
  const double dsq = d0 * d0 + d1 * d1 + d2 * d2;
  if (!(dsq < P.rc2)) return false;
  const double d = sqrt(dsq);
  const double temp = P.c * (P.rc - d) / P.horizon;
  const double cf0 = -(temp * vn * d0 / d), cf1 = -(temp * vn * d1 / d), cf2 = -(temp * vn * d2 / d);
  const double nf0 = temp * vc * d0 / d, nf1 = temp * vc * d1 / d, nf2 = temp * vc * d2 / d;
  fc[0] = cf0; fc[1] = cf1; fc[2] = cf2;
  if (BOTH) { fn[0] = nf0; fn[1] = nf1; fn[2] = nf2; }
  if (P.mu != 0.0) {
    const double n0 = d0 / d, n1 = d1 / d, n2 = d2 / d;
    const double cn = V[0] * n0 + V[1] * n1 + V[2] * n2;
    const double nbn = v[0] * n0 + v[1] * n1 + v[2] * n2;
    const double cp0 = V[0] - cn * n0, cp1 = V[1] - cn * n1, cp2 = V[2] - cn * n2;
    const double np0 = v[0] - nbn * n0, np1 = v[1] - nbn * n1, np2 = v[2] - nbn * n2;
    const double m0 = 0.5 * (cp0 + np0), m1 = 0.5 * (cp1 + np1), m2 = 0.5 * (cp2 + np2);
    const double cr0 = cp0 - m0, cr1 = cp1 - m1, cr2 = cp2 - m2;
    const double ncr = sqrt(cr0 * cr0 + cr1 * cr1 + cr2 * cr2);
    const double ncf = sqrt(cf0 * cf0 + cf1 * cf1 + cf2 * cf2);
    if (ncr != 0.0) {
      fc[0] = cf0 + -P.mu * ncf * cr0 / ncr;
      fc[1] = cf1 + -P.mu * ncf * cr1 / ncr;
      fc[2] = cf2 + -P.mu * ncf * cr2 / ncr;
    }
    if (BOTH) {
      const double nr0 = np0 - m0, nr1 = np1 - m1, nr2 = np2 - m2;
      const double nnr = sqrt(nr0 * nr0 + nr1 * nr1 + nr2 * nr2);
      const double nnf = sqrt(nf0 * nf0 + nf1 * nf1 + nf2 * nf2);
      if (nnr != 0.0) {
        fn[0] = nf0 + -P.mu * nnf * nr0 / nnr;
        fn[1] = nf1 + -P.mu * nnf * nr1 / nnr;
        fn[2] = nf2 + -P.mu * nnf * nr2 / nnr;
      }
    }
  }
  return true;
}

// Explicit-run contact force (internal order) of the points with contacts
// (the others keep the zero written at the search): each point gathers twice
// its own side of every pair of its (symmetric) list, kGatherLanes lanes per
// point (thread t), lane l taking entries l, l + kGatherLanes, ..., then a
// lane-tree sum. Positions as the reference forms them, y = (x + u) + dt v,
// from the record of the step's start (u) and the half-step velocity v (dt = 0
// at the initial evaluation). Whole waves call it.
__device__ __forceinline__ void contact_gather(const ContactGather& a, int t) {
  const int k = t / kGatherLanes, lane = t % kGatherLanes;
  const bool valid = k < a.nact;
  const int i = valid ? a.act[k] : 0;
  double f[3] = {0.0, 0.0, 0.0};
  if (valid) {
    const long long e0 = a.off[i], e1 = a.off[i + 1];
    double X[3], V[3];
    for (int l = 0; l < 3; l++) {
      V[l] = a.v[3 * i + l];
      X[l] = (a.x[3 * i + l] + a.rec[i].u[l] * a.q) + a.dt * V[l];
    }
    const double vc = a.vol[i];
    for (long long e = e0 + lane; e < e1; e += kGatherLanes) {
      const int j = a.list[e];
      double Y[3], W[3], fc[3], fn[3];
      for (int l = 0; l < 3; l++) {
        W[l] = a.v[3 * j + l];
        Y[l] = (a.x[3 * j + l] + a.rec[j].u[l] * a.q) + a.dt * W[l];
      }
      if (contact_pair<false>(a.P, X, V, vc, Y, W, a.vol[j], fc, fn))
        for (int l = 0; l < 3; l++) f[l] += fc[l];
    }
  }
  // every lane takes part in the shuffles (the group of a point is aligned)
  for (int m = kGatherLanes / 2; m >= 1; m >>= 1)
    for (int l = 0; l < 3; l++) f[l] += __shfl_xor(f[l], m, kGatherLanes);
  if (valid && lane == 0)
    for (int l = 0; l < 3; l++) a.fout[3 * i + l] = 2.0 * f[l];
}

}  // namespace dev
}  // namespace pdg
