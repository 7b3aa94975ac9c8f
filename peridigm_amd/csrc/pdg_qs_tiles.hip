// LDS-tiled FP64 bond passes of the quasi-static path: dilatation, residual
// force, and the tangent's two passes (derivative of the dilatation, then of
// the force) over the Hilbert tiles of the explicit path.
//
// One workgroup owns a tile: it stages its halo's records in LDS as arrays of
// 16-byte slots, and groups of G lanes own the tile's nodes. Lanes reading
// distinct residues of 16 halo slots, which the tiles' bond order provides,
// meet distinct LDS banks, as in the explicit passes.
//
// The untiled kernels gather 80 to 112 bytes a bond through L1 and L2 and are
// bound by those gathers' latency; here HBM and L2 see each halo record once
// per tile and a 2-byte index a bond. Bound by FP64 issue (about 70
// instructions a bond in the tangent's force pass), LDS reads and, on small meshes, by
// the launch and the two rounds of loads before the bond loop. One tangent
// product, dilatation + force pass, against the untiled kernels:
//   3,000-node bar:     5.9 + 6.5 us   (9.5 + 10.5)
//   24,000-node bar:   11.0 + 13.3 us  (32 + 41)
//   200,000-node bar:  57 + 76 us      (223 + 313)
// Records as one 80- to 112-byte structure a node instead of arrays measured
// 61 + 125 us on the last (each lane's load then touches a line of its own,
// and 112 bytes leave one workgroup to a CU in the force pass).
//
// Bond arithmetic, in units of L: X = x_j - x_i, D = u_j - u_i, Y = X + D.
// One reciprocal square root t = 1/sqrt(|X|^2 |Y|^2) gives both quantities
// that the formulas need,
//   g = zeta/|Y| = |X|^2 t   and   1/|Y|^2 = g t,
// where the untiled kernels take two square roots and a division. With
// q = beta theta (less the thermal term), a = alpha_i + alpha_j and
// S = T/|Y| = w [(q_i + q_j) g + a e/|Y|]:
//   d theta_i = 3/m_i sum w V_j g Y.dY,
//   df_i = sum V_j ([w g (dq_i + dq_j) + (w a - S) (Y.dY)/|Y|^2] Y + S dY).
// e/|Y| is 1 - g in the tangent, where it is a geometric term of the order of
// the strain, and (|Y|^2 - |X|^2)/|Y|^2 / (1 + g) in the residual, with
// |Y|^2 - |X|^2 = D.(2X + D), which has no cancellation.

#include <algorithm>

#include "pdg_device.hpp"
#include "pdg_qs_tiles.hpp"

namespace pdg {
namespace {

using namespace dev;

constexpr int WG = kTileThreads;

__device__ __forceinline__ int tile_of_block(int bid, int ntiles) {
  const int per = (ntiles + 7) >> 3;  // a contiguous run of tiles per XCD
  return (bid & 7) * per + (bid >> 3);
}
inline unsigned tile_blocks(int ntiles) { return 8u * (unsigned)((ntiles + 7) >> 3); }

// 1/sqrt(a) and 1/a from the hardware estimates (relative error below 2^-20)
// and one third-order step, which cubes that error.
__device__ __forceinline__ double rsqrt64(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double e = fma(-(a * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double rcp64(double a) {
  const double r = __builtin_amdgcn_rcp(a);
  const double e = fma(-a, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// Influence function of a bond with squared length z2 (lengths in units of
// L). The reciprocals depend on the horizon alone, so they leave the loops.
template <int INFL>
__device__ __forceinline__ double omega64(double z2, double hhat) {
  if (INFL == PDG_INFLUENCE_ONE) return 1.0;
  if (INFL == PDG_INFLUENCE_PARABOLIC_DECAY) {
    const double zeta = sqrt(z2);
    if (zeta > hhat) return 0.0;
    const double s = zeta * (1.0 / hhat);
    return s < 0.5 ? 1.0 : -4.0 * s * s + 4.0 * s;
  }
  return exp(z2 * (-1.0 / (hhat * hhat * 0.4 * 0.4)));
}

// Sum over a node's lanes: its group of G, and with two groups a node the one
// in the neighbouring row of 16.
template <int G, int HV>
__device__ __forceinline__ double lanes_sum(double v) {
  v = group_sum64<G>(v);
  if (HV == 2) v += __shfl_xor(v, 16);
  return v;
}

// What a pass does with a bond. QP_CG is QP_DTHETA with a direction that the
// staging forms. QP_DTHETA3 and QP_DFORCE3 take three directions at once, the
// k-th of them w's component k along axis k (0 along the others): the probes
// of the two-level preconditioner's set-up. They share the geometry and the
// records of one direction; only the sums differ, three and nine.
enum { QP_THETA, QP_DTHETA, QP_FORCE, QP_DFORCE, QP_CG, QP_DTHETA3, QP_DFORCE3 };
template <int PASS>
constexpr bool is_dtheta() { return PASS == QP_DTHETA || PASS == QP_CG || PASS == QP_DTHETA3; }
template <int PASS>
constexpr bool is_dforce() { return PASS == QP_DFORCE || PASS == QP_DFORCE3; }
template <int PASS>
constexpr bool is_dual() { return is_dtheta<PASS>() || is_dforce<PASS>(); }
template <int PASS>
constexpr int nsums() { return PASS == QP_DFORCE3 ? 9 : 3; }

// LDS arrays of a pass, 16-byte slots of one halo node each, at compile-time
// distances (one byte offset addresses all of them): xu[0..2], then
//   QP_THETA   (V, -)
//   QP_DTHETA, QP_CG  (w0, w1), (w2, V)
//   QP_FORCE   (alpha, q), (V, -)
//   QP_DFORCE  (alpha, q), (w0, w1), (w2, dq), and an array of V unless every
//              node has the same
//   QP_DFORCE3 as QP_DFORCE, with (dq1, dq2) after (w2, dq0).
constexpr int HS = kTileHaloMax;
template <int PASS>
constexpr int units() {
  return PASS == QP_THETA ? 4 : PASS == QP_DFORCE ? 6 : PASS == QP_DFORCE3 ? 7 : 5;
}
template <int PASS, bool UNIV>
constexpr int lds_bytes() { return 16 * HS * units<PASS>() + (is_dforce<PASS>() && !UNIV ? 8 * HS : 0); }

// Workgroups of 512 threads, two to a CU (at most 80 KB of LDS each). The
// tangent's force pass with a volume array takes 83 KB, that of three
// directions 90 or 96: one workgroup to a CU then, of 1,024 threads, each
// node's bonds shared by two lane groups.
template <int PASS, bool UNIV>
constexpr int halves() { return lds_bytes<PASS, UNIV>() > 81920 ? 2 : 1; }

// A halo node's record in registers.
template <int PASS>
struct Rec {
  f64x2 v[units<PASS>()];
  double vj;  // tangent's force passes: V
  __device__ double x(int c) const { return c == 0 ? v[0].x : c == 1 ? v[0].y : v[1].x; }
  __device__ double u(int c) const { return c == 0 ? v[1].y : c == 1 ? v[2].x : v[2].y; }
  __device__ double vol() const {
    return PASS == QP_THETA ? v[3].x : is_dtheta<PASS>() ? v[units<PASS>() - 1].y
           : PASS == QP_FORCE ? v[units<PASS>() - 1].x : vj;
  }
  __device__ double alpha() const { return v[3].x; }  // force passes
  __device__ double q() const { return v[3].y; }      // force passes
  __device__ double w(int c) const {                  // tangent passes
    constexpr int k = is_dforce<PASS>() ? 4 : units<PASS>() - 2;
    return c == 0 ? v[k].x : c == 1 ? v[k].y : v[k + 1].x;
  }
  __device__ double dq(int k = 0) const {             // tangent's force passes
    return k == 0 ? v[5].y : k == 1 ? v[units<PASS>() - 1].x : v[units<PASS>() - 1].y;
  }
};

template <int PASS, bool UNIV>
__device__ __forceinline__ void rec_read(Rec<PASS>& r, const char* lds, int jb) {
#pragma unroll
  for (int k = 0; k < units<PASS>(); k++)
    r.v[k] = *reinterpret_cast<const f64x2*>(lds + 16 * HS * k + jb);
  if (is_dforce<PASS>() && !UNIV)
    r.vj = *reinterpret_cast<const double*>(lds + 16 * HS * units<PASS>() + (jb >> 1));
}

// One bond of a pass, added to the lane's sums s when `ok` (one sum for the
// dilatation passes, three for the force passes, and as many for each of three
// directions). UNIV: without the volume factor, which the caller applies to
// the sums. A masked-out bond may address a slot that was never written, and
// give a NaN, so the sums are selected; with three directions the factors are,
// and the caller passes the node itself as such a bond's neighbour.
template <int PASS, bool UNIV, int INFL, bool LIN>
__device__ __forceinline__ void bond(const Rec<PASS>& me, const Rec<PASS>& nb, double hhat,
                                     double thermal, bool ok, double (&s)[nsums<PASS>()]) {
  const double X0 = nb.x(0) - me.x(0), X1 = nb.x(1) - me.x(1), X2 = nb.x(2) - me.x(2);
  const double z2 = fma(X2, X2, fma(X1, X1, X0 * X0));
  const double wv = UNIV ? omega64<INFL>(z2, hhat) : omega64<INFL>(z2, hhat) * nb.vol();
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  if (is_dual<PASS>()) {
    d0 = nb.w(0) - me.w(0); d1 = nb.w(1) - me.w(1); d2 = nb.w(2) - me.w(2);
  }
  const double D0 = nb.u(0) - me.u(0), D1 = nb.u(1) - me.u(1), D2 = nb.u(2) - me.u(2);
  auto add1 = [&](double f, double v) {
    const double n = fma(f, v, s[0]);
    s[0] = ok ? n : s[0];
  };
  auto add3 = [&](double f, double v0, double v1, double v2) {
    const double n0 = fma(f, v0, s[0]), n1 = fma(f, v1, s[1]), n2 = fma(f, v2, s[2]);
    s[0] = ok ? n0 : s[0];
    s[1] = ok ? n1 : s[1];
    s[2] = ok ? n2 : s[2];
  };
  if (LIN) {
    // theta and force linear in u, the force along the reference bond
    constexpr bool dual = is_dual<PASS>();
    if (PASS == QP_DTHETA3) {
      const double f = ok ? wv : 0.0;
      s[0] = fma(f, X0 * d0, s[0]);
      s[1] = fma(f, X1 * d1, s[1]);
      s[2] = fma(f, X2 * d2, s[2]);
      return;
    }
    if (PASS == QP_DFORCE3) {
      const double ar = (me.alpha() + nb.alpha()) * rcp64(z2);
      const double pr[3] = {X0 * d0, X1 * d1, X2 * d2};
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const double c = ok ? wv * fma(ar, pr[k], me.dq(k) + nb.dq(k)) : 0.0;
        s[(3 * k) % nsums<PASS>()] = fma(c, X0, s[(3 * k) % nsums<PASS>()]);
        s[(3 * k + 1) % nsums<PASS>()] = fma(c, X1, s[(3 * k + 1) % nsums<PASS>()]);
        s[(3 * k + 2) % nsums<PASS>()] = fma(c, X2, s[(3 * k + 2) % nsums<PASS>()]);
      }
      return;
    }
    const double pr = fma(X2, dual ? d2 : D2, fma(X1, dual ? d1 : D1, X0 * (dual ? d0 : D0)));
    if (PASS == QP_THETA || is_dtheta<PASS>()) {
      add1(wv, pr);
    } else {
      const double qs = PASS == QP_FORCE ? me.q() + nb.q() : me.dq() + nb.dq();
      add3(wv * fma(me.alpha() + nb.alpha(), pr * rcp64(z2), qs), X0, X1, X2);
    }
    return;
  }
  const double Y0 = X0 + D0, Y1 = X1 + D1, Y2 = X2 + D2;
  const double yy = fma(Y2, Y2, fma(Y1, Y1, Y0 * Y0));
  // points that the deformation brings to one place: e is -|X| (g then is so
  // large that g / (1 + g) is 1), where the force of such a bond has no direction
  const double t = rsqrt64(PASS == QP_THETA ? fmax(z2 * yy, 1e-300) : z2 * yy);
  double g = z2 * t, ryy = g * t;
  // points that coincide in the reference configuration (rare: one branch of
  // the wave, no selects)
  if (__builtin_amdgcn_ballot_w64(z2 == 0.0)) {
    if (z2 == 0.0) {
      g = 0.0;
      ryy = rcp64(yy);
    }
  }
  if (PASS == QP_THETA) {
    const double dd = fma(D2, X2 + Y2, fma(D1, X1 + Y1, D0 * (X0 + Y0)));
    add1(wv, dd * g * rcp64(1.0 + g) - thermal * z2);
  } else if (PASS == QP_DTHETA3) {
    const double f = ok ? wv * g : 0.0;
    s[0] = fma(f, Y0 * d0, s[0]);
    s[1] = fma(f, Y1 * d1, s[1]);
    s[2] = fma(f, Y2 * d2, s[2]);
  } else if (is_dtheta<PASS>()) {
    add1(wv * g, fma(Y2, d2, fma(Y1, d1, Y0 * d0)));
  } else if (PASS == QP_FORCE) {
    const double dd = fma(D2, X2 + Y2, fma(D1, X1 + Y1, D0 * (X0 + Y0)));
    const double ey = dd * ryy * rcp64(1.0 + g);
    add3(wv * fma(me.alpha() + nb.alpha(), ey, (me.q() + nb.q()) * g), Y0, Y1, Y2);
  } else if (PASS == QP_DFORCE3) {
    const double a = me.alpha() + nb.alpha();
    const double S = fma(a, 1.0 - g, (me.q() + nb.q()) * g);  // over w
    const double sv = ok ? wv * S : 0.0, wo = ok ? wv : 0.0, gw = ok ? g : 0.0;
    const double ar = ok ? (a - S) * ryy : 0.0;
    const double Y[3] = {Y0, Y1, Y2}, d[3] = {d0, d1, d2};
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double c = wo * fma(gw, me.dq(k) + nb.dq(k), ar * (Y[k] * d[k]));
#pragma unroll
      for (int j = 0; j < 3; j++) {
        double& t = s[(3 * k + j) % nsums<PASS>()];
        t = fma(c, Y[j], t);
        if (j == k) t = fma(sv, d[k], t);
      }
    }
  } else {
    const double a = me.alpha() + nb.alpha();
    const double S = fma(a, 1.0 - g, (me.q() + nb.q()) * g);  // over w
    const double yd = fma(Y2, d2, fma(Y1, d1, Y0 * d0));
    const double c = wv * fma(g, me.dq() + nb.dq(), (a - S) * (yd * ryy));
    const double sv = wv * S;
    const double n0 = fma(sv, d0, fma(c, Y0, s[0]));
    const double n1 = fma(sv, d1, fma(c, Y1, s[1]));
    const double n2 = fma(sv, d2, fma(c, Y2, s[2]));
    s[0] = ok ? n0 : s[0];
    s[1] = ok ? n1 : s[1];
    s[2] = ok ? n2 : s[2];
  }
}

// What the pass writes, besides what QsTileArgs holds.
struct QsOut {
  const double* w;  // QP_DTHETA: the direction, QP_CG: z; 3n
  double* out;      // force passes: 3n
  double* out3[2];  // QP_DFORCE3: the second and third direction's
  int all;          // QP_FORCE: prescribed DOFs too
  QsCgStart start;  // QP_CG; QP_DFORCE: start.cg null outside a solve
  double* pq_part;  // QP_DFORCE in a solve
};

// A node group's row: CSR range, then the lane's intact bits (two words,
// shifted down by the lane; bits past the row's end clear) and the local
// indices of its first round.
template <int U>
struct Row {
  int rs, deg, mw;
  unsigned long long in[2];
  int lj[U];
};

template <int U>
__device__ __forceinline__ void row_range(const QsTileArgs& a, int node, int n0, int n1, Row<U>& r) {
  const unsigned nd = (unsigned)(node < n1 ? node : n0);
  r.rs = a.row[nd];
  const int re = a.row[nd + 1u];
  r.mw = a.mw[nd];
  r.deg = node < n1 ? re - r.rs : 0;
}

template <int GB, int U>
__device__ __forceinline__ void row_data(const QsTileArgs& a, int l, Row<U>& r) {
  const unsigned long long* mp = a.mask + (unsigned)r.mw;
  const unsigned short* lp = a.t.lcol + (unsigned)(r.rs + l);
#pragma unroll
  for (int k = 0; k < U; k++) r.lj[k] = lp[k * GB];
#pragma unroll
  for (int w = 0; w < 2; w++) {
    const int left = r.deg - 64 * w;
    const unsigned long long vb = left >= 64 ? ~0ull : (left <= 0 ? 0ull : (1ull << left) - 1ull);
    r.in[w] = (~mp[w] & vb) >> l;
  }
}

// What a pass stages of halo node i.
template <int PASS, bool UNIV>
__device__ __forceinline__ void slot_load(const QsTileArgs& a, const QsOut& o, unsigned i,
                                          Rec<PASS>& r) {
#pragma unroll
  for (int k = 0; k < 3; k++) r.v[k] = a.rec.xu[k][i];
  if (PASS == QP_FORCE || is_dforce<PASS>()) r.v[3] = a.rec.aq[i];
  if (is_dtheta<PASS>()) {
    const double* w = o.w + 3u * i;
    r.v[units<PASS>() - 2] = f64x2{w[0], w[1]};
    r.v[units<PASS>() - 1] = f64x2{w[2], a.vol[i]};
  } else if (is_dforce<PASS>()) {
    r.v[4 % units<PASS>()] = a.rec.wd[0][i];
    r.v[5 % units<PASS>()] = a.rec.wd[1][i];
    if (PASS == QP_DFORCE3) r.v[6 % units<PASS>()] = a.rec.wp[0][i];
    if (!UNIV) r.vj = a.vol[i];
  } else {
    r.v[units<PASS>() - 1] = f64x2{a.vol[i], 0.0};
  }
}

template <int PASS, bool UNIV>
__device__ __forceinline__ void slot_store(char* lds, int h, const Rec<PASS>& r) {
#pragma unroll
  for (int k = 0; k < units<PASS>(); k++)
    *reinterpret_cast<f64x2*>(lds + 16 * (HS * k + h)) = r.v[k];
  if (is_dforce<PASS>() && !UNIV)
    *reinterpret_cast<double*>(lds + 16 * HS * units<PASS>() + 8 * h) = r.vj;
}

// One pass over one tile. A node has HV groups of G lanes; group h's lane l
// takes bonds h G + l, + HV G, ... in the tile's bond order, U of them per
// round so that their LDS reads and the next round's local indices are in
// flight together (two groups of a node sit in neighbouring 16-lane rows, so
// each row still reads what the bond order made conflict-free). Bonds past
// the row's end and broken bonds are computed like the others and selected
// away: a local index past the row's end belongs to a later row or the zero
// padding, so it addresses a slot of the arrays.
// U = 4 in the force pass of the tangent took 77.3 us against 78.9 with 2 and
// 82.4 with 1 on the 200,000-node bar; in the others 4 spills registers and 2
// is as fast.
template <int G, int PASS, bool UNIV, int INFL, bool LIN>
__global__ __launch_bounds__((WG * halves<PASS, UNIV>()), 4) void k_qs_tile(QsTileArgs a, QsOut o) {
  constexpr int HV = halves<PASS, UNIV>();
  constexpr int U = PASS == QP_DFORCE && HV == 1 && INFL == PDG_INFLUENCE_ONE ? 4 : 2;
  __shared__ __align__(16) char lds[lds_bytes<PASS, UNIV>()];
  constexpr int NG = WG / G;
  constexpr int T = WG * HV;
  constexpr int GB = G * HV;  // bonds of a node per step
  constexpr int kHaloRounds = (kTileHaloMax + T - 1) / T;
  __shared__ double sums[PASS == QP_CG ? 2 * T / 64 : PASS == QP_DFORCE ? T / 64 : 1];
  const int tile = tile_of_block(blockIdx.x, a.t.ntiles);
  if (tile >= a.t.ntiles) return;
  // launches after the end of a solve return at once
  if ((PASS == QP_CG || PASS == QP_DFORCE) && o.start.cg && o.start.cg->done) return;
  const int n0 = a.t.tile_start[tile], n1 = a.t.tile_start[tile + 1];
  const int h0 = a.t.halo_off[tile], hn = min(a.t.halo_off[tile + 1] - h0, HS);
  const int own = a.t.own_off[tile];
  const int l = (threadIdx.x & (G - 1)) + (HV == 2 ? ((threadIdx.x >> 4) & 1) * G : 0);
  const int grp = HV == 2 ? (threadIdx.x >> 5) * (16 / G) + (threadIdx.x & 15) / G : threadIdx.x / G;
  // Two phases of loads, each in flight together: the halo's node ids and the
  // first round's CSR ranges, then the records, mask words and local indices
  // they address. All unconditional (a thread without a slot or a node reads
  // the tile's first).
  int idx[kHaloRounds];
#pragma unroll
  for (int r = 0; r < kHaloRounds; r++) {
    const int h = threadIdx.x + r * T;
    idx[r] = a.t.halo[(unsigned)(h0 + (h < hn ? h : 0))];
  }
  Row<U> rw;
  row_range(a, n0 + grp, n0, n1, rw);
  row_data<GB, U>(a, l, rw);
  double beta = 0.0;
  bool any = false;  // QP_DTHETA3, QP_DFORCE3: a direction that is not 0
#pragma unroll
  for (int r = 0; r < kHaloRounds; r++) {
    if (r > 0 && r * T >= hn) break;
    Rec<PASS> v;
    const unsigned i = (unsigned)idx[r];
    slot_load<PASS, UNIV>(a, o, i, v);
    if (PASS == QP_DTHETA3 || PASS == QP_DFORCE3) {
      any = any || v.w(0) != 0.0 || v.w(1) != 0.0 || v.w(2) != 0.0;
      if (PASS == QP_DFORCE3) any = any || v.dq(0) != 0.0 || v.dq(1) != 0.0 || v.dq(2) != 0.0;
    }
    if (PASS == QP_CG) {
      const f64x2 p0 = a.rec.wp[0][i], p1 = a.rec.wp[1][i];
      if (r == 0 && cg_start<T>(o.start, sums, beta)) return;
      if (beta != 0.0) {  // the first direction is z
        f64x2 &w0 = v.v[units<PASS>() - 2], &w1 = v.v[units<PASS>() - 1];
        w0.x = fma(beta, p0.x, w0.x);
        w0.y = fma(beta, p0.y, w0.y);
        w1.x = fma(beta, p1.x, w1.x);
      }
    }
    const int h = threadIdx.x + r * T;
    if (h < hn) slot_store<PASS, UNIV>(lds, h, v);
  }
  if (PASS == QP_DTHETA3 || PASS == QP_DFORCE3) {
    // A probe is 0 on most of the mesh: a tile whose halo it does not reach
    // has zero images and skips its bonds (set-up of 480 functions on the
    // 200,000-node bar 15.6 -> 12.6 ms).
    if (!__syncthreads_or(any)) {
      for (int q = threadIdx.x; q < n1 - n0; q += T) {
        const unsigned nd = (unsigned)(n0 + q);
        if (PASS == QP_DTHETA3) {
          a.rec.wd[0][nd] = a.rec.wd[1][nd] = a.rec.wp[0][nd] = f64x2{0.0, 0.0};
        } else {
          for (int c = 0; c < 9; c++) (c < 3 ? o.out : o.out3[c / 3 - 1])[3u * nd + (unsigned)(c % 3)] = 0.0;
        }
      }
      return;
    }
  } else {
    __syncthreads();
  }
  double pq = 0.0;  // QP_DFORCE: this thread's part of w.Kw
  for (int base = n0; base < n1; base += NG) {
    const int node = base + grp;
    const bool valid = node < n1;
    const int nd = valid ? node : n0;
    if (base != n0) {
      row_range(a, node, n0, n1, rw);
      row_data<GB, U>(a, l, rw);
    }
    const int deg = rw.deg;
    const unsigned short* lp = a.t.lcol + (unsigned)(rw.rs + l);
    Rec<PASS> me;
    rec_read<PASS, UNIV>(me, lds, kLdsSlot * (own + (nd - n0)));
    double thermal = 0.0;
    if (PASS == QP_THETA && a.dT) thermal = a.alphaT * a.dT[(unsigned)nd];
    // nodes of a tile are ordered by descending degree: the wave's first
    // group has the largest
    const int rounds = (__builtin_amdgcn_readfirstlane(deg) + GB * U - 1) / (GB * U);
    double s[nsums<PASS>()];
#pragma unroll
    for (int k = 0; k < nsums<PASS>(); k++) s[k] = 0.0;
    int (&lj)[U] = rw.lj;
    for (int c = 0; c < rounds; c++) {
      int ln[U];
      const unsigned short* np = lp + min(c + 1, rounds - 1) * (GB * U);
#pragma unroll
      for (int k = 0; k < U; k++) ln[k] = np[k * GB];
      const int b0 = c * (GB * U);
      const unsigned long long bits = (b0 < 64 ? rw.in[0] : rw.in[1]) >> (b0 & 63);
      const unsigned half[2] = {(unsigned)bits, (unsigned)(bits >> 32)};
#pragma unroll
      for (int k = 0; k < U; k++) {
        Rec<PASS> nb;
        const bool ok = (half[(k * GB) >> 5] & (1u << ((k * GB) & 31))) != 0u;
        // where not the sums but the factors are selected, a masked-out bond
        // must read finite values: its node's own slot
        constexpr bool own_slot = PASS == QP_DTHETA3 || PASS == QP_DFORCE3;
        rec_read<PASS, UNIV>(nb, lds, own_slot && !ok ? kLdsSlot * (own + (nd - n0)) : lj[k]);
        bond<PASS, UNIV, INFL, LIN>(me, nb, a.hhat, thermal, ok, s);
      }
#pragma unroll
      for (int k = 0; k < U; k++) lj[k] = ln[k];
    }
    if (PASS == QP_DTHETA3) {
      const double s0 = lanes_sum<G, HV>(s[0]), s1 = lanes_sum<G, HV>(s[1]), s2 = lanes_sum<G, HV>(s[2]);
      if (!valid || l != 0) continue;
      const double m = a.m[(unsigned)node];
      const double c = (m > 0.0 ? 3.0 / m : 0.0) * (UNIV ? a.vol1 : 1.0);
      const double f = a.L * a.beta[(unsigned)node] * (c * a.L);
      a.rec.wd[0][(unsigned)node] = f64x2{me.w(0), me.w(1)};
      a.rec.wd[1][(unsigned)node] = f64x2{me.w(2), f * s0};
      a.rec.wp[0][(unsigned)node] = f64x2{f * s1, f * s2};
    } else if (PASS == QP_DFORCE3) {
      double f[3];  // lane l's: direction l
#pragma unroll
      for (int k = 0; k < nsums<PASS>(); k++) {
        const double v = lanes_sum<G, HV>(s[k]);
        f[k % 3] = k < 3 || k / 3 == l ? v : f[k % 3];
      }
      if (!valid || l >= 3) continue;
      const double w = l == 0 ? me.w(0) : (l == 1 ? me.w(1) : me.w(2));
      double* const out = l == 0 ? o.out : o.out3[l - 1];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const unsigned q = 3u * (unsigned)node + (unsigned)k;
        const double wk = k == l ? w : 0.0;
        double kw = a.fixed[q] ? wk : -f[k] * (UNIV ? a.vol1 * a.vol1 : me.vol());
        if (a.damp) kw += a.damp[q] * wk;
        out[q] = kw;
      }
    } else if (PASS == QP_THETA || is_dtheta<PASS>()) {
      const double sum = lanes_sum<G, HV>(s[0]);
      if (!valid || l != 0) continue;
      const double m = a.m[(unsigned)node];
      const double c = (m > 0.0 ? 3.0 / m : 0.0) * (UNIV ? a.vol1 : 1.0);
      if (PASS == QP_THETA) {
        const double th = c * (a.L * a.L) * sum;
        a.theta[(unsigned)node] = th;
        double q = a.beta[(unsigned)node] * th;
        if (a.dT) q -= thermal * a.alpha[(unsigned)node];
        a.rec.aq[(unsigned)node].y = q;
      } else {
        const double dq = a.L * (a.beta[(unsigned)node] * (c * a.L * sum));
        a.rec.wd[0][(unsigned)node] = f64x2{me.w(0), me.w(1)};
        a.rec.wd[1][(unsigned)node] = f64x2{me.w(2), dq};
      }
    } else {
      const double f0 = lanes_sum<G, HV>(s[0]), f1 = lanes_sum<G, HV>(s[1]), f2 = lanes_sum<G, HV>(s[2]);
      if (!valid || l >= 3) continue;
      const double f = (l == 0 ? f0 : (l == 1 ? f1 : f2)) * (UNIV ? a.vol1 * a.vol1 : me.vol());
      const unsigned q = 3u * (unsigned)node + (unsigned)l;
      const bool fx = a.fixed[q] != 0;
      if (PASS == QP_FORCE) {
        o.out[q] = fx && !o.all ? 0.0 : a.L * f;
      } else {
        const double w = l == 0 ? me.w(0) : (l == 1 ? me.w(1) : me.w(2));
        double kw = fx ? w : -f;
        if (a.damp) kw += a.damp[q] * w;
        o.out[q] = kw;
        pq += w * kw;
      }
    }
  }
  if (PASS == QP_DFORCE && o.start.cg) {
    pq = wave_sum64(pq);
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = pq;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int k = 0; k < T / 64; k++) t += sums[k];
      o.pq_part[tile] = t;
    }
  }
}

__global__ __launch_bounds__(256) void k_qs_pack(QsTileArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  const double iL = 1.0 / a.L;  // exact
  const double* x = a.x + 3 * (size_t)i;
  const double* u = a.u + 3 * (size_t)i;
  a.rec.xu[0][i] = f64x2{x[0] * iL, x[1] * iL};
  a.rec.xu[1][i] = f64x2{x[2] * iL, u[0] * iL};
  a.rec.xu[2][i] = f64x2{u[1] * iL, u[2] * iL};
  a.rec.aq[i] = f64x2{a.alpha[i], 0.0};
}

// G lanes per node: at least enough that one round covers a tile, and at most
// 16, the width of the LDS service groups that the bond order is made for
// (wider settings run as 16 and loop over the tile's nodes).
template <int PASS, bool UNIV, int INFL, bool LIN>
hipError_t launch_g(const QsTileArgs& a, const QsOut& o, int lanes, hipStream_t s) {
  const dim3 grid(tile_blocks(a.t.ntiles)), blk(WG * halves<PASS, UNIV>());
  if (lanes <= 4) hipLaunchKernelGGL((k_qs_tile<4, PASS, UNIV, INFL, LIN>), grid, blk, 0, s, a, o);
  else if (lanes == 8) hipLaunchKernelGGL((k_qs_tile<8, PASS, UNIV, INFL, LIN>), grid, blk, 0, s, a, o);
  else hipLaunchKernelGGL((k_qs_tile<16, PASS, UNIV, INFL, LIN>), grid, blk, 0, s, a, o);
  return hipGetLastError();
}

template <int PASS, int INFL, bool LIN>
hipError_t launch_v(const QsTileArgs& a, const QsOut& o, int lanes, hipStream_t s) {
  if (a.vol1 > 0.0) return launch_g<PASS, true, INFL, LIN>(a, o, lanes, s);
  return launch_g<PASS, false, INFL, LIN>(a, o, lanes, s);
}

template <int PASS>
hipError_t launch(const QsTileArgs& a, const QsOut& o, int lanes, hipStream_t s) {
  if (a.t.ntiles <= 0) return hipErrorInvalidValue;
  if (a.influence == PDG_INFLUENCE_ONE)
    return a.linear ? launch_v<PASS, 0, true>(a, o, lanes, s) : launch_v<PASS, 0, false>(a, o, lanes, s);
  if (a.influence == PDG_INFLUENCE_PARABOLIC_DECAY)
    return a.linear ? launch_v<PASS, 1, true>(a, o, lanes, s) : launch_v<PASS, 1, false>(a, o, lanes, s);
  return a.linear ? launch_v<PASS, 2, true>(a, o, lanes, s) : launch_v<PASS, 2, false>(a, o, lanes, s);
}

}  // namespace

hipError_t launch_qs_state(const QsTileArgs& a, int lanes, hipStream_t s) {
  hipLaunchKernelGGL(k_qs_pack, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, s, a);
  return launch<QP_THETA>(a, QsOut{}, lanes, s);
}

hipError_t launch_qs_residual(const QsTileArgs& a, bool all, double* out, int lanes,
                              hipStream_t s) {
  QsOut o{};
  o.out = out;
  o.all = all ? 1 : 0;
  return launch<QP_FORCE>(a, o, lanes, s);
}

hipError_t launch_qs_tangent(const QsTileArgs& a, const double* w, double* out, int lanes,
                             hipStream_t s) {
  QsOut o{};
  o.w = w;
  o.out = out;
  hipError_t e = launch<QP_DTHETA>(a, o, lanes, s);
  return e == hipSuccess ? launch<QP_DFORCE>(a, o, lanes, s) : e;
}

hipError_t launch_qs_tangent3(const QsTileArgs& a, const double* w, double* const (&out)[3],
                              int lanes, hipStream_t s) {
  QsOut o{};
  o.w = w;
  o.out = out[0];
  o.out3[0] = out[1];
  o.out3[1] = out[2];
  hipError_t e = launch<QP_DTHETA3>(a, o, lanes, s);
  return e == hipSuccess ? launch<QP_DFORCE3>(a, o, lanes, s) : e;
}

hipError_t launch_qs_tangent_cg(const QsTileArgs& a, const QsCgStart& start, const double* z,
                                double* out, double* pq_part, int lanes, hipStream_t s) {
  QsOut o{};
  o.w = z;
  o.out = out;
  o.start = start;
  o.pq_part = pq_part;
  hipError_t e = launch<QP_CG>(a, o, lanes, s);
  return e == hipSuccess ? launch<QP_DFORCE>(a, o, lanes, s) : e;
}

}  // namespace pdg
