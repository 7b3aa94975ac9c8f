// LDS-tiled FP64 bond passes of the quasi-static path (pdg_qs_tiles.hip).
#pragma once

#include "pdg_qs_cg.hpp"

namespace pdg {

typedef double f64x2 __attribute__((ext_vector_type(2)));

// Node records of the tiled passes as arrays of 16-byte units (n entries
// each), so that a tile's halo, sorted node ids in mostly contiguous runs, is
// read in whole cache lines: xu[0..2] = (x0, x1), (x2, u0), (u1, u2) in units
// of the context's power-of-two length L (exact); aq = (alpha, q) with
// alpha = 15 mu / m and q = beta theta (less alphaT alpha dT with thermal
// strains), the node's share of a bond's dilatation term; wd = (w0, w1),
// (w2, L beta dtheta): the direction of a tangent product and the derivative
// of the dilatation term along it.
struct QsRecords {
  f64x2* xu[3];
  f64x2* aq;
  f64x2* wd[2];
  f64x2* wp[2];  // the previous direction of a conjugate-gradient solve
};

struct QsTileArgs {
  TileArgs t;
  int n;
  const int* row;
  const int* mw;
  const unsigned long long* mask;
  const double* m;
  const double* beta;
  const double* alpha;
  const double* vol;
  double vol1;  // > 0: every node's volume
  const double* x;  // 3n
  const double* u;  // 3n
  double L, hhat;   // length scale, horizon / L
  int influence;
  bool linear;       // linearized LPS
  const double* dT;  // temperature change per node, or null
  double alphaT;
  const signed char* fixed;
  const double* damp;  // 3n, added to the tangent's diagonal, or null
  QsRecords rec;
  double* theta;
};

// Fills the records xu and aq and theta from x, u and the node constants:
// what the launches below read.
hipError_t launch_qs_state(const QsTileArgs& a, int lanes, hipStream_t s);
// out = f V at that state, 0 on prescribed DOFs unless `all`.
hipError_t launch_qs_residual(const QsTileArgs& a, bool all, double* out, int lanes,
                              hipStream_t s);
// out = K w at that state (w on prescribed DOFs); w: 3n.
hipError_t launch_qs_tangent(const QsTileArgs& a, const double* w, double* out, int lanes,
                             hipStream_t s);

// out[k] = K (w's component k along axis k) for the three axes; uses the
// records wp.
hipError_t launch_qs_tangent3(const QsTileArgs& a, const double* w, double* const (&out)[3],
                              int lanes, hipStream_t s);

// The same product for a conjugate-gradient iteration: w = z + beta wp (the
// records wp) with beta and the decision to stop from `start`, w into the
// records wd; pq_part[t] is tile t's part of w.Kw.
hipError_t launch_qs_tangent_cg(const QsTileArgs& a, const QsCgStart& start, const double* z,
                                double* out, double* pq_part, int lanes, hipStream_t s);

}  // namespace pdg
