// Neighbour-list construction on the device. Integer results from FP64
// predicates evaluated with the reference's operation order and no FMA
// contraction (built with -ffp-contract=off), so the lists are bit-identical
// to the reference builders.
//   QuickGrid lattice:  src/io/mesh_input/quick_grid/QuickGrid.cxx:160-165,
//                       :243-253, :394-408, :510-647
//   radius search:      src/io/Peridigm_ZoltanSearchTree.cpp:236-246 (<= R^2),
//                       rows sorted by id (src/io/pdneigh/NeighborhoodList.cxx:705)
//   finite-plane filter: src/io/pdneigh/BondFilter.cxx:59-153

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <vector>

#include "pdg_internal.hpp"

namespace {

struct QGrid {
  int n[3];
  int hw[3];
  const double* c[3];
  double r;
  int spherical;
};

__device__ __forceinline__ void qg_window(int i, int h, int n, int& s, int& e) {
  s = i > h ? i - h : 0;
  e = i < (n - h) ? i + h + 1 : n;
}

// Visits the candidate window of lattice cell (i,j,k) in kk -> jj -> ii order.
template <bool FILL>
__global__ __launch_bounds__(256) void k_quickgrid(QGrid g, long long* __restrict__ count,
                                                   const long long* __restrict__ head,
                                                   int* __restrict__ nlist) {
  const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long N = (long long)g.n[0] * g.n[1] * g.n[2];
  if (gid >= N) return;
  const int i = (int)(gid % g.n[0]);
  const int j = (int)((gid / g.n[0]) % g.n[1]);
  const int k = (int)(gid / ((long long)g.n[0] * g.n[1]));
  const double p0 = g.c[0][i], p1 = g.c[1][j], p2 = g.c[2][k];
  int xs, xe, ys, ye, zs, ze;
  qg_window(i, g.hw[0], g.n[0], xs, xe);
  qg_window(j, g.hw[1], g.n[1], ys, ye);
  qg_window(k, g.hw[2], g.n[2], zs, ze);
  long long out = FILL ? head[gid] + 1 : 0;
  int cnt = 0;
  for (int kk = zs; kk < ze; kk++)
    for (int jj = ys; jj < ye; jj++)
      for (int ii = xs; ii < xe; ii++) {
        if (ii == i && jj == j && kk == k) continue;
        bool in = true;
        if (g.spherical) {
          const double dx = p0 - g.c[0][ii];
          const double dy = p1 - g.c[1][jj];
          const double dz = p2 - g.c[2][kk];
          in = dx * dx + dy * dy + dz * dz - g.r * g.r < 0.0;
        }
        if (in) {
          if (FILL) nlist[out++] = (int)(ii + (long long)jj * g.n[0] + (long long)kk * g.n[0] * g.n[1]);
          cnt++;
        }
      }
  if (FILL) nlist[head[gid]] = cnt;
  else count[gid] = cnt;
}

__global__ void k_head(long long n, const long long* __restrict__ excl, long long* __restrict__ head) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) head[i] = excl[i] + i;
}

// ---- radius search --------------------------------------------------------
struct RGrid {
  double lo[3];
  double cs;
  int nc[3];
  double R2;
};

__device__ __forceinline__ int cell_coord(double x, double lo, double cs, int nc) {
  int c = (int)floor((x - lo) / cs);
  return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

// Partial bounding boxes (lo, hi per block) of the points; NaNs drop out, as
// in the comparisons of a host loop.
constexpr int kBoxBlocks = 64;
__global__ __launch_bounds__(256) void k_box(int n, const double* __restrict__ x,
                                             double* __restrict__ part) {
  __shared__ double sh[4][6];
  double b[6] = {DBL_MAX, DBL_MAX, DBL_MAX, -DBL_MAX, -DBL_MAX, -DBL_MAX};
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    for (int d = 0; d < 3; d++) {
      b[d] = fmin(b[d], x[3 * (size_t)i + d]);
      b[3 + d] = fmax(b[3 + d], x[3 * (size_t)i + d]);
    }
  for (int o = 32; o > 0; o >>= 1)
    for (int d = 0; d < 3; d++) {
      b[d] = fmin(b[d], __shfl_xor(b[d], o));
      b[3 + d] = fmax(b[3 + d], __shfl_xor(b[3 + d], o));
    }
  if ((threadIdx.x & 63) == 0)
    for (int d = 0; d < 6; d++) sh[threadIdx.x >> 6][d] = b[d];
  __syncthreads();
  if (threadIdx.x < 6) {
    const int d = threadIdx.x;
    double v = sh[0][d];
    for (int w = 1; w < 4; w++) v = d < 3 ? fmin(v, sh[w][d]) : fmax(v, sh[w][d]);
    part[6 * blockIdx.x + d] = v;
  }
}

__device__ __forceinline__ void cell_of(const RGrid& g, double X0, double X1, double X2, int (&c)[3]) {
  c[0] = cell_coord(X0, g.lo[0], g.cs, g.nc[0]);
  c[1] = cell_coord(X1, g.lo[1], g.cs, g.nc[1]);
  c[2] = cell_coord(X2, g.lo[2], g.cs, g.nc[2]);
}

// Points of each cell, then (after a scan into `begin`) the points and their
// positions by cell; the order inside a cell is left to the atomics, since
// the rows are sorted at the end.
__global__ void k_cell_count(int n, const double* __restrict__ x, RGrid g, int* __restrict__ cell,
                             int* __restrict__ count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int c[3];
  cell_of(g, x[3 * (size_t)i], x[3 * (size_t)i + 1], x[3 * (size_t)i + 2], c);
  const int id = (c[2] * g.nc[1] + c[1]) * g.nc[0] + c[0];
  cell[i] = id;
  atomicAdd(&count[id], 1);
}

// count: what is left of each cell (counted down to 0)
__global__ void k_cell_scatter(int n, const double* __restrict__ x, const int* __restrict__ cell,
                               const int* __restrict__ begin, int* __restrict__ count,
                               int* __restrict__ sidx, double* __restrict__ xs) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int q = begin[cell[i]] + atomicSub(&count[cell[i]], 1) - 1;
  sidx[q] = i;
  for (int d = 0; d < 3; d++) xs[3 * (size_t)q + d] = x[3 * (size_t)i + d];
}

// FinitePlane::bondIntersectInfinitePlane + bondIntersect (tolerance 1e-15),
// FinitePlaneFilter::filterBonds with p0 = the point, p1 = its neighbour.
__device__ bool plane_cuts(const double* pl, const double* p0, const double* p1) {
  const double* nrm = pl;
  const double* r0 = pl + 3;
  const double* ub = pl + 6;
  const double b = pl[9], a = pl[10];
  double ua[3];
  ua[0] = -ub[2] * nrm[1] + ub[1] * nrm[2];
  ua[1] = ub[2] * nrm[0] - ub[0] * nrm[2];
  ua[2] = -ub[1] * nrm[0] + ub[0] * nrm[1];
  const double numerator =
      (r0[0] - p0[0]) * nrm[0] + (r0[1] - p0[1]) * nrm[1] + (r0[2] - p0[2]) * nrm[2];
  const double denominator =
      (p1[0] - p0[0]) * nrm[0] + (p1[1] - p0[1]) * nrm[1] + (p1[2] - p0[2]) * nrm[2];
  double t;
  if (fabs(denominator) < 1.0e-14) t = DBL_MAX;
  else t = numerator / denominator;
  if (!(t >= 0.0 && t <= 1.0)) return false;
  double xi[3];
  xi[0] = p0[0] + t * (p1[0] - p0[0]);
  xi[1] = p0[1] + t * (p1[1] - p0[1]);
  xi[2] = p0[2] + t * (p1[2] - p0[2]);
  const double zero = 1.0e-15;
  const double one = 1.0 + zero;
  const double dr0 = xi[0] - r0[0], dr1 = xi[1] - r0[1], dr2 = xi[2] - r0[2];
  const double aa = dr0 * ua[0] + dr1 * ua[1] + dr2 * ua[2];
  const double bb = dr0 * ub[0] + dr1 * ub[1] + dr2 * ub[2];
  return -zero < aa && aa / a < one && -zero < bb && bb / b < one;
}

// One wave per point, in cell order: candidates from the 27 surrounding cells
// (nine runs of the cell order, three cells along x each), 64 at a time;
// membership by the predicate alone. The lanes' hits are packed into the
// wave's LDS row, the packed row is filtered by the planes, and FILL ranks its
// ids (unique: an id's place is the number of smaller ones) and writes the
// row in order. COUNT only counts. Rows that outgrow the LDS row are flushed
// in pieces: counted, or written unsorted to `spill` for k_spilled_rows.
// Against a thread per point (whose lanes walk cells of different lengths),
// a radix sort of 64-bit (row, id) keys and per-bond kernels for the planes
// and the compaction, 160,000 points with 13.7M bonds and one plane: 0.23 ms
// to count and 0.33 ms to fill (the kernels before took 1.9 and 2.7 ms). Bound
// by instruction issue: two in three candidates fail the distance test, and
// ranking a row of 122 takes 244 broadcast compares a lane.
constexpr int kRowCap = 512;
using pdg::kGroupWaves;
struct NearArgs {
  int n;
  RGrid g;
  const double* xs;
  const int* sidx;
  const int* begin;
  int nplanes;
  const double* planes;
  long long* count;
  const long long* off;  // FILL: kept bonds of the rows before
  int* nlist;
  int* big;              // COUNT: set when any row was flushed
  int* spill;            // FILL, if so: the flushed rows, unsorted
  int* flushed;          // FILL, if so: which rows they are
};

// Orders the wave's LDS accesses before and after it.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool FILL>
__global__ __launch_bounds__(64 * kGroupWaves) void k_near(NearArgs a) {
  __shared__ __align__(16) int rows[kGroupWaves][kRowCap + 68];
  const int lane = threadIdx.x & 63;
  int* const row = rows[threadIdx.x >> 6];
  const long long at = pdg::wave_index();
  if (at >= a.n) return;  // whole waves: no barrier below
  const int t = (int)at;
  const int i = a.sidx[t];
  const double P[3] = {a.xs[3 * (size_t)t], a.xs[3 * (size_t)t + 1], a.xs[3 * (size_t)t + 2]};
  int c[3];
  cell_of(a.g, P[0], P[1], P[2], c);
  const unsigned long long below = (1ull << lane) - 1ull;
  int nb = 0;            // entries of the LDS row: sorted positions, then (filtered) ids
  long long total = 0;   // kept so far (flushed pieces)
  bool flushed = false;
  // filters the LDS row by the planes and turns positions into ids
  auto filter = [&]() {
    int kept = 0;
    for (int e0 = 0; e0 < nb; e0 += 64) {
      const bool have = e0 + lane < nb;
      const int q = have ? row[e0 + lane] : t;
      bool keep = have;
      if (a.nplanes > 0 && have) {
        const double Q[3] = {a.xs[3 * (size_t)q], a.xs[3 * (size_t)q + 1], a.xs[3 * (size_t)q + 2]};
        for (int p = 0; p < a.nplanes && keep; p++) keep = !plane_cuts(a.planes + 11 * p, P, Q);
      }
      const int id = a.sidx[q];
      const unsigned long long m = __ballot(keep);
      wave_sync();
      if (keep) row[kept + __popcll(m & below)] = id;  // never past what was read
      wave_sync();
      kept += __popcll(m);
    }
    nb = kept;
  };
  auto flush = [&]() {
    filter();
    if (FILL)
      for (int e = lane; e < nb; e += 64) a.spill[a.off[i] + total + e] = row[e];
    total += nb;
    nb = 0;
    flushed = true;
  };
  for (int dz = -1; dz <= 1; dz++) {
    const int cz = c[2] + dz;
    if (cz < 0 || cz >= a.g.nc[2]) continue;
    for (int dy = -1; dy <= 1; dy++) {
      const int cy = c[1] + dy;
      if (cy < 0 || cy >= a.g.nc[1]) continue;
      const int first = (cz * a.g.nc[1] + cy) * a.g.nc[0];
      const int s = a.begin[first + max(c[0] - 1, 0)];
      const int e = a.begin[first + min(c[0] + 1, a.g.nc[0] - 1) + 1];
      for (int q0 = s; q0 < e; q0 += 64) {
        const int q = q0 + lane;
        bool hit = false;
        if (q < e && q != t) {
          const double d0 = a.xs[3 * (size_t)q] - P[0], d1 = a.xs[3 * (size_t)q + 1] - P[1],
                       d2 = a.xs[3 * (size_t)q + 2] - P[2];
          hit = d0 * d0 + d1 * d1 + d2 * d2 <= a.g.R2;
        }
        const unsigned long long m = __ballot(hit);
        if (nb > kRowCap) flush();
        if (hit) row[nb + __popcll(m & below)] = q;
        wave_sync();
        nb += __popcll(m);
      }
    }
  }
  if (flushed) flush();
  else if (FILL || a.nplanes > 0) filter();
  if (!FILL) {
    if (lane == 0) {
      a.count[i] = total + nb;
      if (flushed) *a.big = 1;
    }
    return;
  }
  const long long h = a.off[i] + i;
  if (lane == 0) a.nlist[h] = (int)(total + nb);
  if (a.flushed && lane == 0) a.flushed[i] = flushed;
  if (flushed) return;
  // pad to whole groups of four that no id ranks above
  if (lane < 4) row[nb + lane] = INT_MAX;
  wave_sync();
  for (int e = lane; e < nb; e += 64) {
    const int v = row[e];
    int rank = 0;
    for (int k = 0; k < nb; k += 4) {
      const int4 w = *reinterpret_cast<const int4*>(row + k);
      rank += (w.x < v) + (w.y < v) + (w.z < v) + (w.w < v);
    }
    a.nlist[h + 1 + rank] = v;
  }
}

// The flushed rows, sorted from `spill` (a workgroup per row): pieces of up to
// kSortPiece ids in LDS (bitonic, padded to a power of two), and where a row has
// more than one, each id then goes to its place in its piece plus the number of
// smaller ids in the others (ids are unique). Work per row of m ids is about
// m log^2 m; counting the smaller ones for every id took m^2: lists of 22,000
// points that are all in each other's radius 1.82 s, with this 0.30 (a radix sort
// of all bonds, before, 0.64).
constexpr int kSortPiece = 4096;
constexpr int kSortThreads = 256;
__global__ __launch_bounds__(kSortThreads) void k_spilled_rows(
    int n, const long long* __restrict__ count, const long long* __restrict__ off, int* spill,
    const int* __restrict__ flushed, int* __restrict__ nlist) {
  __shared__ int a[kSortPiece];
  const long long at = pdg::group_index();
  if (at >= n || !flushed[at]) return;
  const long long m = count[at];
  int* const r = spill + off[at];
  int* const out = nlist + off[at] + at + 1;
  for (long long p0 = 0; p0 < m; p0 += kSortPiece) {
    const int len = (int)min((long long)kSortPiece, m - p0);
    int size = 64;
    while (size < len) size *= 2;
    for (int e = threadIdx.x; e < size; e += kSortThreads) a[e] = e < len ? r[p0 + e] : INT_MAX;
    for (int k = 2; k <= size; k *= 2)
      for (int j = k / 2; j > 0; j /= 2) {
        __syncthreads();
        for (int t = threadIdx.x; t < size / 2; t += kSortThreads) {
          const int e = 2 * t - (t & (j - 1));  // e's bit j is clear
          const int x = a[e], y = a[e + j];
          if ((x > y) == ((e & k) == 0)) {
            a[e] = y;
            a[e + j] = x;
          }
        }
      }
    __syncthreads();
    int* const to = m <= kSortPiece ? out : r + p0;
    for (int e = threadIdx.x; e < len; e += kSortThreads) to[e] = a[e];
    __syncthreads();
  }
  if (m <= kSortPiece) return;
  for (long long e = threadIdx.x; e < m; e += kSortThreads) {
    const int v = r[e];
    const long long own = e / kSortPiece;
    long long place = e - own * kSortPiece;
    for (long long p = 0; p * kSortPiece < m; p++) {
      if (p == own) continue;
      const int* const s = r + p * kSortPiece;
      int lo = 0;  // ids of the piece below v
      for (int hi = (int)min((long long)kSortPiece, m - p * kSortPiece); lo < hi;) {
        const int mid = (lo + hi) / 2;
        if (s[mid] < v) lo = mid + 1;
        else hi = mid;
      }
      place += lo;
    }
    out[place] = v;
  }
}

template <class T>
struct DevBuf {
  T* p = nullptr;
  hipError_t alloc(size_t n) { return hipMalloc((void**)&p, std::max<size_t>(n, 1) * sizeof(T)); }
  ~DevBuf() { if (p) (void)hipFree(p); }
};

#define PDG_CK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) return PDG_E_HIP; } while (0)

int exclusive_scan(const long long* in, long long* out, long long n, hipStream_t s) {
  size_t bytes = 0;
  PDG_CK(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n, s));
  DevBuf<char> tmp;
  PDG_CK(tmp.alloc(bytes));
  PDG_CK(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, in, out, (int)n, s));
  return PDG_OK;
}

}  // namespace

extern "C" {

int pdg_quickgrid(int nx, int ny, int nz, const double origin[3], const double length[3],
                  double horizon, int spherical, double* x, double* volume, int* nlist,
                  long long* listSize) {
  if (nx <= 0 || ny <= 0 || nz <= 0 || !origin || !length || !listSize) return PDG_E_ARG;
  const long long N = (long long)nx * ny * nz;
  if (N >= (1ll << 31)) return PDG_E_UNSUPPORTED;
  const int n[3] = {nx, ny, nz};
  std::vector<double> c[3];
  int hw[3];
  for (int d = 0; d < 3; d++) {
    // Spec1D::getCellSize, getDiscretization (centres by accumulation),
    // getCellNeighborhoodSize (window in cells, rounded, clamped).
    const double cs = length[d] / n[d];
    c[d].resize(n[d]);
    double p = origin[d] + cs / 2.0;
    for (int i = 0; i < n[d]; p += cs, i++) c[d][i] = p;
    const double dCx = horizon / (cs * 1.0);
    size_t nC = static_cast<size_t>(dCx);
    if (std::abs(dCx - nC) >= .5) nC += 1;
    if (nC > (size_t)n[d]) nC = n[d];
    hw[d] = (int)nC;
  }
  hipStream_t s = nullptr;
  DevBuf<double> dc0, dc1, dc2;
  DevBuf<long long> cnt, excl, head;
  PDG_CK(dc0.alloc(nx)); PDG_CK(dc1.alloc(ny)); PDG_CK(dc2.alloc(nz));
  PDG_CK(hipMemcpy(dc0.p, c[0].data(), 8 * nx, hipMemcpyHostToDevice));
  PDG_CK(hipMemcpy(dc1.p, c[1].data(), 8 * ny, hipMemcpyHostToDevice));
  PDG_CK(hipMemcpy(dc2.p, c[2].data(), 8 * nz, hipMemcpyHostToDevice));
  QGrid g;
  for (int d = 0; d < 3; d++) { g.n[d] = n[d]; g.hw[d] = hw[d]; }
  g.c[0] = dc0.p; g.c[1] = dc1.p; g.c[2] = dc2.p;
  g.r = horizon;
  g.spherical = spherical;
  PDG_CK(cnt.alloc(N)); PDG_CK(excl.alloc(N)); PDG_CK(head.alloc(N));
  const unsigned blocks = (unsigned)((N + 255) / 256);
  hipLaunchKernelGGL((k_quickgrid<false>), dim3(blocks), dim3(256), 0, s, g, cnt.p, nullptr, nullptr);
  PDG_CK(hipGetLastError());
  int rc = exclusive_scan(cnt.p, excl.p, N, s);
  if (rc) return rc;
  long long lastc = 0, laste = 0;
  PDG_CK(hipMemcpy(&lastc, cnt.p + N - 1, 8, hipMemcpyDeviceToHost));
  PDG_CK(hipMemcpy(&laste, excl.p + N - 1, 8, hipMemcpyDeviceToHost));
  const long long size = laste + lastc + N;
  const long long cap = *listSize;
  *listSize = size;
  if (x)
    for (long long gid = 0; gid < N; gid++) {
      const int i = (int)(gid % nx), j = (int)((gid / nx) % ny), k = (int)(gid / ((long long)nx * ny));
      x[3 * gid] = c[0][i]; x[3 * gid + 1] = c[1][j]; x[3 * gid + 2] = c[2][k];
    }
  if (volume) {
    const double cv = (length[0] / nx) * (length[1] / ny) * (length[2] / nz);
    for (long long gid = 0; gid < N; gid++) volume[gid] = cv;
  }
  if (!nlist) return PDG_OK;
  if (cap < size) return PDG_E_ARG;
  hipLaunchKernelGGL(k_head, dim3(blocks), dim3(256), 0, s, N, excl.p, head.p);
  DevBuf<int> dl;
  PDG_CK(dl.alloc(size));
  hipLaunchKernelGGL((k_quickgrid<true>), dim3(blocks), dim3(256), 0, s, g, nullptr, head.p, dl.p);
  PDG_CK(hipGetLastError());
  PDG_CK(hipMemcpy(nlist, dl.p, 4 * size, hipMemcpyDeviceToHost));
  return PDG_OK;
}

int pdg_radius_search(int N, const double* x, double R, int nplanes, const double* planes,
                      int* nlist, long long* listSize) {
  if (N <= 0 || !x || !(R > 0.0) || !listSize || nplanes < 0 || (nplanes > 0 && !planes))
    return PDG_E_ARG;
  hipStream_t s = nullptr;
  const unsigned nb = (unsigned)((N + 255) / 256);
  DevBuf<double> dx, dpl;
  PDG_CK(dx.alloc(6 * (size_t)N + 6 * kBoxBlocks));  // x, sorted positions, boxes
  double* const xs = dx.p + 3 * (size_t)N;
  double* const dbox = xs + 3 * (size_t)N;
  PDG_CK(hipMemcpyAsync(dx.p, x, 24 * (size_t)N, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_box, dim3(kBoxBlocks), dim3(256), 0, s, N, dx.p, dbox);
  double box[6 * kBoxBlocks];
  PDG_CK(hipMemcpy(box, dbox, sizeof(box), hipMemcpyDeviceToHost));
  double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  for (int b = 0; b < kBoxBlocks; b++)
    for (int d = 0; d < 3; d++) {
      lo[d] = std::min(lo[d], box[6 * b + d]);
      hi[d] = std::max(hi[d], box[6 * b + 3 + d]);
    }
  NearArgs a{};
  RGrid& g = a.g;
  g.cs = R * 1.0000001;
  long long ncell = 1;
  for (int d = 0; d < 3; d++) {
    g.lo[d] = lo[d];
    g.nc[d] = std::max(1, (int)std::floor((hi[d] - lo[d]) / g.cs) + 1);
    ncell *= g.nc[d];
  }
  if (ncell > (1ll << 30)) return PDG_E_UNSUPPORTED;
  g.R2 = R * R;
  // cells: counts (one more, 0, for the scan) and first points; points: cell
  // and cell order; the flush flag
  const size_t nc1 = (size_t)ncell + 1, n1 = (size_t)N + 1;
  DevBuf<int> ints;
  PDG_CK(ints.alloc(2 * nc1 + 2 * (size_t)N + 1));
  int* const ccount = ints.p;
  int* const begin = ccount + nc1;
  int* const cell = begin + nc1;
  int* const sidx = cell + N;
  int* const big = sidx + N;
  DevBuf<long long> sums;  // bonds of each row (a 0 after the last) and of the rows before
  PDG_CK(sums.alloc(2 * n1));
  long long* const count = sums.p;
  long long* const off = count + n1;
  // one workspace for both scans
  size_t bytes = 0, b2 = 0;
  PDG_CK(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, ccount, begin, (int)nc1, s));
  PDG_CK(hipcub::DeviceScan::ExclusiveSum(nullptr, b2, count, off, (int)n1, s));
  bytes = std::max(bytes, b2);
  DevBuf<char> tmp;
  PDG_CK(tmp.alloc(bytes));
  PDG_CK(dpl.alloc(std::max(1, 11 * nplanes)));
  if (nplanes > 0) PDG_CK(hipMemcpyAsync(dpl.p, planes, 88 * (size_t)nplanes, hipMemcpyHostToDevice, s));
  PDG_CK(hipMemsetAsync(ccount, 0, 4 * nc1, s));
  PDG_CK(hipMemsetAsync(big, 0, 4, s));
  PDG_CK(hipMemsetAsync(count + N, 0, 8, s));
  hipLaunchKernelGGL(k_cell_count, dim3(nb), dim3(256), 0, s, N, dx.p, g, cell, ccount);
  PDG_CK(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, ccount, begin, (int)nc1, s));
  hipLaunchKernelGGL(k_cell_scatter, dim3(nb), dim3(256), 0, s, N, dx.p, cell, begin, ccount, sidx, xs);
  a.n = N; a.xs = xs; a.sidx = sidx; a.begin = begin; a.nplanes = nplanes; a.planes = dpl.p;
  a.count = count; a.off = off; a.big = big;
  const dim3 nw = pdg::wave_grid(N);
  hipLaunchKernelGGL(k_near<false>, nw, dim3(64 * kGroupWaves), 0, s, a);
  PDG_CK(hipGetLastError());
  PDG_CK(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, count, off, (int)n1, s));
  long long B = 0;
  int hbig = 0;
  PDG_CK(hipMemcpyAsync(&hbig, big, 4, hipMemcpyDeviceToHost, s));
  PDG_CK(hipMemcpy(&B, off + N, 8, hipMemcpyDeviceToHost));
  PDG_CK(hipStreamSynchronize(s));
  const long long size = B + N;
  const long long cap = *listSize;
  *listSize = size;
  if (!nlist) return PDG_OK;
  if (cap < size) return PDG_E_ARG;
  DevBuf<int> list, spill;
  PDG_CK(list.alloc(size));
  if (hbig) PDG_CK(spill.alloc((size_t)B + (size_t)N));
  a.nlist = list.p;
  a.spill = spill.p;
  a.flushed = hbig ? spill.p + B : nullptr;
  hipLaunchKernelGGL(k_near<true>, nw, dim3(64 * kGroupWaves), 0, s, a);
  if (hbig)
    hipLaunchKernelGGL(k_spilled_rows, pdg::group_grid(N), dim3(kSortThreads), 0, s, N, count, off, spill.p,
                       a.flushed, list.p);
  PDG_CK(hipGetLastError());
  PDG_CK(hipMemcpy(nlist, list.p, 4 * size, hipMemcpyDeviceToHost));
  return PDG_OK;
}

}  // extern "C"
