// Short-range contact: the contact search of the current configuration and
// the short-range force contact model.
//
// Reference: src/core/Peridigm_ContactManager.cpp:700-750 (contactSearch: a
// neighbourhood search of the current positions within the contact search
// radius, the point's bonded neighbours dropped, broken or not),
// src/contact/Peridigm_ShortRangeForceContactModel.cpp:98-258 (computeForce)
// and src/core/Peridigm.cpp:1468-1472, 1515-1524, 1559-1565 (the search at
// every step whose number is a multiple of the search frequency, before the
// first half kick; the contact force added to the internal force before the
// acceleration).
//
// Search: positions hashed into a spatial grid of cells no smaller than the
// search radius (2^k buckets, k the smallest with 2^k >= 2N), points sorted by
// bucket. A point looks up the buckets of its 27 surrounding cells, meeting
// every point in them once; the distance predicate alone decides membership,
// as in the reference. The counting pass tests no bonds per candidate: a point's
// contact count is its points within the radius less its bonded neighbours
// within it, both under one predicate, so the difference is exact. Only the
// points with contacts are walked again to write their rows, finding bonded
// neighbours by binary search in the point's bond row (kept sorted in a copy
// of the bond list).
//
// Force: the search list is symmetric (j lists i exactly when i lists j: the
// squared distance and the bond lists are symmetric), and the reference adds
// the same pair term to a point once from its own list and once from its
// neighbour's, so the explicit run gathers 2 x (the point's side of every
// pair) with no atomics. The drop-in call takes any list and scatters both
// sides, as the reference does, with FP64 atomic adds.

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "pdg_contact_dev.hpp"
#include "pdg_ctx.hpp"

namespace pdg {

struct ContactState {
  double R = 0.0;       // search radius
  double rc = 0.0;      // contact radius
  double ks = 0.0;      // spring constant
  double mu = 0.0;      // friction coefficient
  double c = 0.0;       // 9 ks / (pi horizon^4)
  int freq = 1;         // search frequency (steps)
  long long step = 0;   // steps since the last initial evaluation
  bool built = false;   // a search list exists
  unsigned nbits = 1;   // log2 of the bucket count
  double inv_cs = 0.0;  // 1 / cell size
  // device, internal order unless stated
  double* y = nullptr;            // 3n positions of the search
  double* fc = nullptr;           // 3n contact force density of the last evaluation
  int* bcol = nullptr;            // bond list, each row ascending (rows: Ctx::d_row)
  int *key = nullptr, *idx = nullptr, *skey = nullptr, *sidx = nullptr;
  int *bstart = nullptr, *bend = nullptr;
  long long *cnt = nullptr, *off = nullptr;  // n+1 each (cnt[n] = 0)
  int* list = nullptr;
  long long cap = 0, size = 0;
  int* act = nullptr;   // n: points with contacts
  int* nact_d = nullptr;
  int nact = 0;
  double* ys = nullptr;  // 3n positions in bucket order
  unsigned char* code = nullptr;  // n: cell codes in bucket order
  int* over = nullptr;   // n: points with contacts, in any order (the filling pass)
  int* nover_d = nullptr;
  void* tmp = nullptr;
  size_t tmp_bytes = 0;
  // drop-in call buffers (reference order)
  double *vref = nullptr, *dv = nullptr, *dfc = nullptr;
  long long* dhead = nullptr;
  int* dlist = nullptr;
  long long dcap = 0;
};

namespace {

// Cell coordinate of one position component; huge or non-finite values are
// clamped (clamping keeps cells of points within one cell size of each other
// adjacent).
__device__ __forceinline__ int cell_of(double p, double inv_cs) {
  double c = floor(p * inv_cs);
  c = fmin(fmax(c, -1073741824.0), 1073741824.0);
  return (int)c;
}

__device__ __forceinline__ unsigned bucket_of(int a, int b, int c, unsigned mask) {
  return ((unsigned)a * 73856093u ^ (unsigned)b * 19349663u ^ (unsigned)c * 83492791u) & mask;
}

__global__ void k_contact_y(int n, const NodeRec* __restrict__ rec, const double* __restrict__ x,
                            double q, double* __restrict__ y) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 3 * n) return;
  const int k = t / 3, l = t - 3 * k;
  y[t] = x[t] + rec[k].u[l] * q;
}

__global__ void k_contact_y_perm(int n, const double* __restrict__ yref, const int* __restrict__ perm,
                                 double* __restrict__ y) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 3 * n) return;
  const int k = t / 3, l = t - 3 * k;
  y[t] = yref[3 * (size_t)perm[k] + l];
}

__global__ void k_contact_keys(int n, const double* __restrict__ y, double inv_cs, unsigned mask,
                               int* __restrict__ key, int* __restrict__ idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int a = cell_of(y[3 * i], inv_cs), b = cell_of(y[3 * i + 1], inv_cs),
            c = cell_of(y[3 * i + 2], inv_cs);
  key[i] = (int)bucket_of(a, b, c, mask);
  idx[i] = i;
}

__global__ void k_fill_int(long long n, int* __restrict__ p, int v) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

__global__ void k_fill_f64(long long n, double* __restrict__ p) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.0;
}

// Two low bits of each cell coordinate: tells a cell from its 26 neighbours.
__device__ __forceinline__ unsigned cell_code(int a, int b, int c) {
  return (unsigned)(a & 3) | (unsigned)(b & 3) << 2 | (unsigned)(c & 3) << 4;
}

// Bucket-ordered copy of the positions: a bucket's candidates are then read
// contiguously. Also each point's cell code.
__global__ void k_contact_ys(int n, const int* __restrict__ sidx, const double* __restrict__ y,
                             double inv_cs, double* __restrict__ ys,
                             unsigned char* __restrict__ code) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const double* p = y + 3 * (size_t)sidx[q];
  const double y0 = p[0], y1 = p[1], y2 = p[2];
  double* o = ys + 3 * (size_t)q;
  o[0] = y0; o[1] = y1; o[2] = y2;
  code[q] = (unsigned char)cell_code(cell_of(y0, inv_cs), cell_of(y1, inv_cs), cell_of(y2, inv_cs));
}

__global__ void k_bucket_bounds(int n, const int* __restrict__ skey, int* __restrict__ bstart,
                                int* __restrict__ bend) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int b = skey[q];
  if (q == 0 || skey[q - 1] != b) bstart[b] = q;
  if (q == n - 1 || skey[q + 1] != b) bend[b] = q + 1;
}

// The search predicate, |p - P|^2 <= R^2 with the differences taken as
// p - P: every kernel that decides membership evaluates it this way, so the
// counting and filling passes agree bit for bit.
__device__ __forceinline__ bool within(const double* __restrict__ p, double P0, double P1,
                                       double P2, double R2) {
  const double d0 = p[0] - P0, d1 = p[1] - P1, d2 = p[2] - P2;
  return d0 * d0 + d1 * d1 + d2 * d2 <= R2;
}

// Contact count of every point: the points within the search radius in the
// buckets of its 27 cells, less its bonded neighbours within the radius.
// Every bonded neighbour within the radius is one of the former, so the
// count is that of the unbonded ones, with no bond test per candidate. A
// point within the radius lies in one of the 27 cells, and its cell code says
// in which: it counts only where that cell is looked up, so it counts once
// even when two of the cells share a bucket.
// kCountLanes threads per point in bucket order (t: the sorted position), so
// a wave's lanes mostly walk the same buckets; lane l of a point reads the
// bounds of the buckets l, l + kCountLanes, ... ahead (all in flight) and takes
// every kCountLanes-th candidate and bond. A thread per point, which removed
// shared buckets by comparing all pairs of the 27, left 2.4 waves to a SIMD on
// 160,000 points and waited for its reads: 261 us, now 171 (209 with 2 lanes, 184 to 187 with 8 and 16).
constexpr int kCountLanes = 4;
__global__ __launch_bounds__(256) void k_contact_count(
    int n, const double* __restrict__ ys, const unsigned char* __restrict__ code,
    const int* __restrict__ sidx, const double* __restrict__ y, double R2, double inv_cs,
    unsigned mask, const int* __restrict__ bstart, const int* __restrict__ bend,
    const int* __restrict__ brow, const int* __restrict__ bcol, long long* __restrict__ cnt,
    int* __restrict__ nover, int* __restrict__ over) {
  constexpr int G = kCountLanes, NB = (27 + G - 1) / G;
  const int t = (blockIdx.x * 256 + threadIdx.x) / G, l = threadIdx.x & (G - 1);
  const bool valid = t < n;
  const int tt = valid ? t : 0;
  const int i = sidx[tt];
  const double Y0 = ys[3 * (size_t)tt], Y1 = ys[3 * (size_t)tt + 1], Y2 = ys[3 * (size_t)tt + 2];
  const int a = cell_of(Y0, inv_cs), b = cell_of(Y1, inv_cs), c = cell_of(Y2, inv_cs);
  int s[NB], e[NB];
#pragma unroll
  for (int r = 0; r < NB; r++) {
    const int k = min(r * G + l, 26);
    const unsigned bk = bucket_of(a + k % 3 - 1, b + (k / 3) % 3 - 1, c + k / 9 - 1, mask);
    s[r] = bstart[bk];
    e[r] = bend[bk];
  }
  int count = 0;
#pragma unroll
  for (int k = 0; k < 27; k++) {
    const int q0 = __shfl(s[k / G], k % G, G), q1 = __shfl(e[k / G], k % G, G);
    const unsigned want = cell_code(a + k % 3 - 1, b + (k / 3) % 3 - 1, c + k / 9 - 1);
    int q = q0 + l;
    for (; q + G < q1; q += 2 * G) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int p = q + u * G;
        count += (p != t && within(ys + 3 * (size_t)p, Y0, Y1, Y2, R2) && code[p] == want) ? 1 : 0;
      }
    }
    if (q < q1)
      count += (q != t && within(ys + 3 * (size_t)q, Y0, Y1, Y2, R2) && code[q] == want) ? 1 : 0;
  }
  const int r1 = brow[i + 1];
  int bo = brow[i] + l;
  for (; bo + 3 * G < r1; bo += 4 * G) {
    int jj[4];
#pragma unroll
    for (int u = 0; u < 4; u++) jj[u] = bcol[bo + u * G];
#pragma unroll
    for (int u = 0; u < 4; u++) count -= within(y + 3 * (size_t)jj[u], Y0, Y1, Y2, R2) ? 1 : 0;
  }
  for (; bo < r1; bo += G) count -= within(y + 3 * (size_t)bcol[bo], Y0, Y1, Y2, R2) ? 1 : 0;
  for (int o = G / 2; o > 0; o >>= 1) count += __shfl_xor(count, o, G);
  if (!valid || l != 0) return;
  cnt[i] = count;
  if (count > 0) over[atomicAdd(nover, 1)] = i;
}

// Contact rows of the points of `pts` (those with contacts; their number in
// *npts), written at off[i] in visit order: the buckets of the 27 cells in
// turn, each distinct one once (a bucket that two of the cells share is left
// out the second time), each point's within the radius kept unless bonded.
// A wave per point: lane k looks up bucket k; the candidates of all buckets,
// numbered through by a running sum of the buckets' sizes, go 64 at a time;
// hits search the point's sorted bond row (in LDS up to kRowLds bonds) and the
// rest are packed behind those before them. Few points have contacts, so a
// thread per point left the GPU to a handful of waves, each walking some 300
// candidates: 469 us on the notch of a 160,000-node plate, now 15.
constexpr int kRowLds = 256;
__global__ __launch_bounds__(64 * kGroupWaves) void k_contact_rows(
    const int* __restrict__ npts, const int* __restrict__ pts, const double* __restrict__ y,
    const double* __restrict__ ys, double R2, double inv_cs, unsigned mask,
    const int* __restrict__ bstart, const int* __restrict__ bend, const int* __restrict__ sidx,
    const int* __restrict__ brow, const int* __restrict__ bcol, const long long* __restrict__ off,
    int* __restrict__ list) {
  __shared__ int rows[kGroupWaves][kRowLds];
  __shared__ int first[kGroupWaves][28], base[kGroupWaves][28];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long t = wave_index();
  if (t >= *npts) return;  // whole waves: no barrier below
  const int i = pts[t];
  const double Y0 = y[3 * (size_t)i], Y1 = y[3 * (size_t)i + 1], Y2 = y[3 * (size_t)i + 2];
  const int a = cell_of(Y0, inv_cs), b = cell_of(Y1, inv_cs), c = cell_of(Y2, inv_cs);
  const int r0 = brow[i], deg = brow[i + 1] - r0;
  const bool in_lds = deg <= kRowLds;
  if (in_lds)
    for (int k = lane; k < deg; k += 64) rows[w][k] = bcol[r0 + k];
  const int k = min(lane, 26);
  const unsigned bk = bucket_of(a + k % 3 - 1, b + (k / 3) % 3 - 1, c + k / 9 - 1, mask);
  bool dup = lane >= 27;
  for (int p = 0; p < 26; p++) {
    const unsigned o = __shfl(bk, p);  // every lane takes part
    dup |= p < lane && o == bk;
  }
  const int s = bstart[bk];
  const int size = dup ? 0 : bend[bk] - s;
  int sum = size;  // inclusive running sum over the lanes
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(sum, o);
    if (lane >= o) sum += v;
  }
  if (lane < 28) {
    first[w][lane] = sum - size;        // number of the bucket's first candidate
    base[w][lane] = s - (sum - size);   // its place less that number
  }
  const int total = __shfl(sum, 63);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  int* const out = list + off[i];
  int count = 0;
  for (int f0 = 0; f0 < total; f0 += 64) {
    const int f = f0 + lane;
    // the last bucket whose first number is <= f (empty buckets share theirs
    // with the next one, so the last is the one that holds f)
    int g = 0;
    for (int step = 16; step > 0; step >>= 1)
      if (g + step < 27 && first[w][g + step] <= f) g += step;
    const int q = f < total ? base[w][g] + f : 0;
    const int j = sidx[q];
    bool keep = f < total && j != i && within(ys + 3 * (size_t)q, Y0, Y1, Y2, R2);
    if (__ballot(keep)) {
      int pos = 0;  // the last entry <= j, if any
      for (int m = deg; m > 1;) {
        const int half = m >> 1;
        const int v = in_lds ? rows[w][pos + half] : bcol[r0 + pos + half];
        pos = v <= j ? pos + half : pos;
        m -= half;
      }
      if (deg > 0) keep = keep && (in_lds ? rows[w][pos] : bcol[r0 + pos]) != j;
    }
    const unsigned long long m = __ballot(keep);
    if (keep) out[count + __popcll(m & ((1ull << lane) - 1ull))] = j;
    count += __popcll(m);
  }
}

// Points with a non-empty contact list, appended in any order (each point's
// force is computed on its own, so the order does not reach the results).
__global__ void k_contact_active(int n, const long long* __restrict__ cnt, int* __restrict__ nact,
                                 int* __restrict__ act) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || cnt[i] == 0) return;
  act[atomicAdd(nact, 1)] = i;
}

// The explicit run's contact force by itself (untiled runs, per-pass timing).
__global__ __launch_bounds__(256) void k_contact_gather(ContactGather a) {
  dev::contact_gather(a, blockIdx.x * 256 + threadIdx.x);
}

// Drop-in contact force (reference order, any list): both sides of every
// listed pair, the neighbour's through FP64 atomic adds.
__global__ __launch_bounds__(256) void k_contact_scatter(
    int n, const double* __restrict__ y, const double* __restrict__ v,
    const double* __restrict__ vol, const long long* __restrict__ head,
    const int* __restrict__ list, PairParams P, double* __restrict__ fout) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long long h = head[i];
  const int nn = list[h];
  if (nn <= 0) return;
  double X[3], V[3];
  for (int l = 0; l < 3; l++) { X[l] = y[3 * i + l]; V[l] = v[3 * i + l]; }
  const double vc = vol[i];
  double f[3] = {0.0, 0.0, 0.0};
  for (int k = 0; k < nn; k++) {
    const int j = list[h + 1 + k];
    double Y[3], W[3], fc[3], fn[3];
    for (int l = 0; l < 3; l++) { Y[l] = y[3 * j + l]; W[l] = v[3 * j + l]; }
    if (dev::contact_pair<true>(P, X, V, vc, Y, W, vol[j], fc, fn)) {
      for (int l = 0; l < 3; l++) {
        f[l] += fc[l];
        unsafeAtomicAdd(fout + 3 * (size_t)j + l, fn[l]);
      }
    }
  }
  for (int l = 0; l < 3; l++) unsafeAtomicAdd(fout + 3 * (size_t)i + l, f[l]);
}

inline unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

PairParams pair_params(const Ctx* c) {
  const ContactState* S = c->contact;
  return PairParams{S->rc, S->rc * S->rc, S->c, c->horizon, S->mu};
}

template <class T>
int grow(Ctx* c, T*& p, long long& cap, long long need, const char* what) {
  if (need <= cap && p) return PDG_OK;
  if (p) (void)hipFree(p);
  p = nullptr;
  cap = 0;
  const long long n = std::max<long long>(need + need / 4, 1024);
  int rc = c->hip(hipMalloc((void**)&p, (size_t)n * sizeof(T)), what);
  if (!rc) cap = n;
  return rc;
}

int tmp_reserve(Ctx* c, size_t bytes) {
  ContactState* S = c->contact;
  if (bytes <= S->tmp_bytes && S->tmp) return PDG_OK;
  if (S->tmp) (void)hipFree(S->tmp);
  S->tmp = nullptr;
  S->tmp_bytes = 0;
  int rc = c->hip(hipMalloc(&S->tmp, std::max<size_t>(bytes, 256)), "alloc contact temp");
  if (!rc) S->tmp_bytes = std::max<size_t>(bytes, 256);
  return rc;
}

// The contact list of the positions in S->y (internal order) into S->off /
// S->list; synchronises the stream once (the list size). For an explicit run
// (`run`) also the list of points with contacts and a zero contact force.
int search(Ctx* c, bool run) {
  ContactState* S = c->contact;
  const int N = c->N;
  hipStream_t s = c->stream;
  const unsigned nb = blocks_for(N);
  const unsigned mask = (1u << S->nbits) - 1u;
  hipLaunchKernelGGL(k_contact_keys, dim3(nb), dim3(256), 0, s, N, S->y, S->inv_cs, mask, S->key,
                     S->idx);
  size_t bytes = 0;
  int rc = c->hip(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, S->key, S->skey, S->idx,
                                                     S->sidx, N, 0, (int)S->nbits, s),
                  "contact sort size");
  if (!rc) rc = tmp_reserve(c, bytes);
  if (!rc) rc = c->hip(hipcub::DeviceRadixSort::SortPairs(S->tmp, bytes, S->key, S->skey, S->idx,
                                                          S->sidx, N, 0, (int)S->nbits, s),
                       "contact sort");
  if (rc) return rc;
  const long long T = 1ll << S->nbits;
  hipLaunchKernelGGL(k_fill_int, dim3(blocks_for(T)), dim3(256), 0, s, T, S->bstart, 0);
  hipLaunchKernelGGL(k_fill_int, dim3(blocks_for(T)), dim3(256), 0, s, T, S->bend, 0);
  hipLaunchKernelGGL(k_bucket_bounds, dim3(nb), dim3(256), 0, s, N, S->skey, S->bstart, S->bend);
  hipLaunchKernelGGL(k_contact_ys, dim3(nb), dim3(256), 0, s, N, S->sidx, S->y, S->inv_cs, S->ys,
                     S->code);
  const double R2 = S->R * S->R;
  hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, s, 1ll, S->nover_d, 0);
  hipLaunchKernelGGL(k_contact_count, dim3(blocks_for((long long)N * kCountLanes)), dim3(256), 0, s,
                     N, S->ys, S->code, S->sidx, S->y, R2,
                     S->inv_cs, mask, S->bstart, S->bend, c->d_row, S->bcol, S->cnt, S->nover_d,
                     S->over);
  rc = c->hip(hipGetLastError(), "contact count");
  bytes = 0;
  if (!rc) rc = c->hip(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, S->cnt, S->off, N + 1, s),
                       "contact scan size");
  if (!rc) rc = tmp_reserve(c, bytes);
  if (!rc) rc = c->hip(hipcub::DeviceScan::ExclusiveSum(S->tmp, bytes, S->cnt, S->off, N + 1, s),
                       "contact scan");
  // points with contacts; the force of every other point is zero until the
  // next search
  if (!rc && run) {
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, s, 1ll, S->nact_d, 0);
    hipLaunchKernelGGL(k_contact_active, dim3(nb), dim3(256), 0, s, N, S->cnt, S->nact_d, S->act);
    hipLaunchKernelGGL(k_fill_f64, dim3(blocks_for(3ll * N)), dim3(256), 0, s, 3ll * N, S->fc);
  }
  long long total = 0;
  int nact = 0;
  if (!rc) rc = c->hip(hipMemcpyAsync(&total, S->off + N, 8, hipMemcpyDeviceToHost, s), "d2h size");
  if (!rc && run) rc = c->hip(hipMemcpyAsync(&nact, S->nact_d, 4, hipMemcpyDeviceToHost, s), "d2h active");
  if (!rc) rc = c->hip(hipStreamSynchronize(s), "sync");
  if (run) S->nact = nact;
  if (!rc) rc = grow(c, S->list, S->cap, total, "alloc contact list");
  if (rc) return rc;
  // the rows of the points with contacts (their number stays on the device:
  // threads past it return at once)
  if (total > 0)
    hipLaunchKernelGGL(k_contact_rows, wave_grid(N), dim3(64 * kGroupWaves), 0, s, S->nover_d, S->over, S->y,
                       S->ys, R2, S->inv_cs, mask, S->bstart, S->bend, S->sidx, c->d_row, S->bcol, S->off,
                       S->list);
  rc = c->hip(hipGetLastError(), "contact fill");
  S->size = total;
  S->built = run;
  return rc;
}

}  // namespace

void Ctx::free_contact() {
  if (!contact) return;
  ContactState* S = contact;
  void* ptrs[] = {S->y, S->fc, S->bcol, S->key, S->idx, S->skey, S->sidx, S->bstart,
                  S->bend, S->cnt, S->off, S->list, S->tmp, S->vref, S->dv, S->dfc,
                  S->dhead, S->dlist, S->act, S->nact_d, S->ys, S->code, S->over, S->nover_d};
  for (void* p : ptrs) if (p) (void)hipFree(p);
  delete S;
  contact = nullptr;
}

bool contact_on(const Ctx* c) { return c->contact != nullptr && c->N > 0; }

const double* contact_force_ptr(const Ctx* c) { return c->contact ? c->contact->fc : nullptr; }

// Step bookkeeping of an explicit run: evaluation k (0: initial) of a run.
// rec_prev holds the displacement at the start of step k (the previous
// evaluation's), rec the initial one at k = 0. Searches, when one is due, in
// the configuration x + u of that displacement; g is the evaluation's contact
// force at y = x + u + dt v, for a launch of either kind.
int contact_step(Ctx* c, int k, double dt, const NodeRec* rec_prev, const NodeRec* rec,
                 ContactGather* g) {
  ContactState* S = c->contact;
  const int N = c->N;
  hipStream_t s = c->stream;
  const NodeRec* const u = k == 0 ? rec : rec_prev;
  S->step = k == 0 ? 0 : S->step + 1;
  if (k == 0 || !S->built || S->step % S->freq == 0) {
    hipLaunchKernelGGL(k_contact_y, dim3(blocks_for(3ll * N)), dim3(256), 0, s, N, u, c->d_x, c->q,
                       S->y);
    int rc = search(c, true);
    if (rc) return rc;
  }
  *g = ContactGather{S->nact, S->act, u, c->d_x, c->q, k == 0 ? 0.0 : dt, c->d_v, c->d_vol,
                     S->off, S->list, pair_params(c), S->fc};
  return PDG_OK;
}

hipError_t launch_contact_gather(const ContactGather& g, hipStream_t s) {
  if (g.nact == 0) return hipSuccess;  // all zero since the search
  hipLaunchKernelGGL(k_contact_gather, dim3(blocks_for((long long)g.nact * kGatherLanes)), dim3(256),
                     0, s, g);
  return hipGetLastError();
}

}  // namespace pdg

using namespace pdg;

extern "C" {

int pdg_set_contact(pdg_ctx* h, double searchRadius, int searchFrequency, double contactRadius,
                    double springConstant, double frictionCoefficient) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  if (!c || !c->have_consts) return PDG_E_ARG;
  if (!(contactRadius > 0.0)) {  // off
    c->free_contact();
    return PDG_OK;
  }
  if (!(searchRadius > 0.0) || searchFrequency < 1 || !std::isfinite(springConstant) ||
      !std::isfinite(frictionCoefficient) || !std::isfinite(searchRadius) ||
      !std::isfinite(contactRadius))
    return c->fail(PDG_E_ARG, "invalid contact parameters");
  if ((long long)c->col.size() != c->B || (int)c->row.size() != c->N + 1)
    return c->fail(PDG_E_ARG, "contact needs the bond lists of the constants");
  (void)hipSetDevice(c->device);
  c->free_contact();
  c->contact = new ContactState();
  ContactState* S = c->contact;
  S->R = searchRadius;
  S->rc = contactRadius;
  S->ks = springConstant;
  S->mu = frictionCoefficient;
  S->freq = searchFrequency;
  const double pi = 3.14159265358979323846;
  const double hz = c->horizon;
  S->c = 9.0 * springConstant / (pi * hz * hz * hz * hz);
  S->inv_cs = 1.0 / (searchRadius * 1.0000001);
  const int N = c->N;
  while ((1ll << S->nbits) < 2ll * std::max(N, 1)) S->nbits++;
  const long long T = 1ll << S->nbits;
  auto A = [&](auto*& p, long long n, const char* what) {
    return c->hip(hipMalloc((void**)&p, (size_t)std::max<long long>(n, 1) * sizeof(*p)), what);
  };
  const long long B = c->B;
  int rc = A(S->y, 3ll * N, "alloc contact y");
  if (!rc) rc = A(S->fc, 3ll * N, "alloc contact f");
  if (!rc) rc = A(S->bcol, B, "alloc contact bonds");
  if (!rc) rc = A(S->key, N, "alloc contact keys");
  if (!rc) rc = A(S->idx, N, "alloc contact keys");
  if (!rc) rc = A(S->skey, N, "alloc contact keys");
  if (!rc) rc = A(S->sidx, N, "alloc contact keys");
  if (!rc) rc = A(S->bstart, T, "alloc contact buckets");
  if (!rc) rc = A(S->bend, T, "alloc contact buckets");
  if (!rc) rc = A(S->cnt, N + 1ll, "alloc contact counts");
  if (!rc) rc = A(S->off, N + 1ll, "alloc contact offsets");
  if (!rc) rc = A(S->vref, N, "alloc contact volumes");
  if (!rc) rc = A(S->act, N, "alloc contact active list");
  if (!rc) rc = A(S->nact_d, 1, "alloc contact active count");
  if (!rc) rc = A(S->ys, 3ll * N, "alloc contact sorted positions");
  if (!rc) rc = A(S->code, N, "alloc contact cell codes");
  if (!rc) rc = A(S->over, N, "alloc contact point list");
  if (!rc) rc = A(S->nover_d, 1, "alloc contact point count");
  if (rc) { c->free_contact(); return rc; }
  // bond rows (internal ids) sorted ascending
  std::vector<int> bc(c->col.begin(), c->col.end());
  for (int k = 0; k < N; k++) std::sort(bc.begin() + c->row[k], bc.begin() + c->row[k + 1]);
  hipStream_t s = c->stream;
  const long long zero = 0;
  if (B > 0) rc = c->hip(hipMemcpyAsync(S->bcol, bc.data(), 4 * (size_t)B, hipMemcpyHostToDevice, s), "h2d bonds");
  if (!rc) rc = c->hip(hipMemcpyAsync(S->cnt + N, &zero, 8, hipMemcpyHostToDevice, s), "h2d zero");
  if (!rc && N > 0) rc = c->hip(hipMemcpyAsync(S->vref, c->vol.data(), 8 * (size_t)N, hipMemcpyHostToDevice, s), "h2d vol");
  if (!rc) hipLaunchKernelGGL(k_fill_f64, dim3(blocks_for(3ll * N)), dim3(256), 0, s, 3ll * N, S->fc);
  if (!rc) rc = c->hip(hipStreamSynchronize(s), "sync");
  if (rc) c->free_contact();
  return rc;
}

int pdg_contact_search(pdg_ctx* h, const double* y, int* contactList, long long* listSize) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  if (!c || !listSize || (c->N > 0 && !y)) return PDG_E_ARG;
  if (!c->contact) return c->fail(PDG_E_ARG, "no contact model (pdg_set_contact)");
  (void)hipSetDevice(c->device);
  ContactState* S = c->contact;
  const int N = c->N;
  hipStream_t s = c->stream;
  int rc = c->hip(hipMemcpyAsync(c->d_y, y, 24 * (size_t)N, hipMemcpyHostToDevice, s), "h2d y");
  if (rc) return rc;
  hipLaunchKernelGGL(k_contact_y_perm, dim3(blocks_for(3ll * N)), dim3(256), 0, s, N, c->d_y,
                     c->d_perm, S->y);
  // the explicit run rebuilds its list from its own state afterwards
  rc = search(c, false);
  if (rc) return rc;
  const long long size = S->size + N;
  const long long cap = *listSize;
  *listSize = size;
  if (!contactList) return PDG_OK;
  if (cap < size) return c->fail(PDG_E_ARG, "contact list capacity too small");
  std::vector<long long> off(N + 1);
  std::vector<int> lst((size_t)S->size);
  rc = c->hip(hipMemcpyAsync(off.data(), S->off, 8 * (size_t)(N + 1), hipMemcpyDeviceToHost, s), "d2h off");
  if (!rc && S->size > 0)
    rc = c->hip(hipMemcpyAsync(lst.data(), S->list, 4 * (size_t)S->size, hipMemcpyDeviceToHost, s), "d2h list");
  if (!rc) rc = c->hip(hipStreamSynchronize(s), "sync");
  if (rc) return rc;
  // reference order, neighbours ascending
  long long p = 0;
  std::vector<int> r;
  for (int g = 0; g < N; g++) {
    const int k = c->iperm[g];
    r.clear();
    for (long long e = off[k]; e < off[k + 1]; e++) r.push_back(c->perm[lst[e]]);
    std::sort(r.begin(), r.end());
    contactList[p++] = (int)r.size();
    for (int j : r) contactList[p++] = j;
  }
  return PDG_OK;
}

int pdg_contact_compute_force(pdg_ctx* h, double dt, const double* y, const double* v,
                              const int* contactList, long long listSize, double* contactForce) {
  (void)dt;
  Ctx* c = reinterpret_cast<Ctx*>(h);
  if (!c || (c->N > 0 && (!y || !v || !contactList || !contactForce))) return PDG_E_ARG;
  if (!c->contact) return c->fail(PDG_E_ARG, "no contact model (pdg_set_contact)");
  const int N = c->N;
  if (N == 0) return PDG_OK;
  // list heads, checked against the stated size and the node range
  std::vector<long long> head(N);
  long long p = 0;
  for (int i = 0; i < N; i++) {
    if (p >= listSize) return c->fail(PDG_E_ARG, "contact list shorter than its counts");
    head[i] = p;
    const int nn = contactList[p];
    if (nn < 0 || p + 1 + nn > listSize) return c->fail(PDG_E_ARG, "contact list shorter than its counts");
    for (int k = 0; k < nn; k++) {
      const int j = contactList[p + 1 + k];
      if (j < 0 || j >= N) return c->fail(PDG_E_ARG, "contact neighbour out of range");
    }
    p += 1 + nn;
  }
  (void)hipSetDevice(c->device);
  ContactState* S = c->contact;
  hipStream_t s = c->stream;
  int rc = PDG_OK;
  if (!S->dv) rc = c->hip(hipMalloc((void**)&S->dv, 24 * (size_t)N), "alloc contact v");
  if (!rc && !S->dfc) rc = c->hip(hipMalloc((void**)&S->dfc, 24 * (size_t)N), "alloc contact f");
  if (!rc && !S->dhead) rc = c->hip(hipMalloc((void**)&S->dhead, 8 * (size_t)N), "alloc contact heads");
  if (!rc) rc = grow(c, S->dlist, S->dcap, p, "alloc contact list");
  // small meshes: everything through the staging buffer as set-up made it, but
  // for a list that does not fit (14 contacts a node)
  const size_t vb = 24 * (size_t)N, hb = 8 * (size_t)N, lb = 4 * (size_t)p;
  char* st = !rc && N <= kHostOrderMax ? c->stage(2 * vb + hb) : nullptr;
  auto up = [&](void* dev, const void* host, size_t bytes, size_t at, const char* what) {
    if (rc) return;
    const void* from = st && at + bytes <= c->h_stage_bytes ? std::memcpy(st + at, host, bytes) : host;
    rc = c->hip(hipMemcpyAsync(dev, from, bytes, hipMemcpyHostToDevice, s), what);
  };
  up(c->d_y, y, vb, 0, "h2d y");
  up(S->dv, v, vb, vb, "h2d v");
  up(S->dhead, head.data(), hb, 2 * vb, "h2d heads");
  up(S->dlist, contactList, lb, 2 * vb + hb, "h2d list");
  if (rc) {
    (void)hipStreamSynchronize(s);
    return rc;
  }
  hipLaunchKernelGGL(k_fill_f64, dim3(blocks_for(3ll * N)), dim3(256), 0, s, 3ll * N, S->dfc);
  hipLaunchKernelGGL(k_contact_scatter, dim3(blocks_for(N)), dim3(256), 0, s, N, c->d_y, S->dv,
                     S->vref, S->dhead, S->dlist, pair_params(c), S->dfc);
  rc = c->hip(hipGetLastError(), "contact force");
  if (!rc) rc = c->hip(hipMemcpyAsync(st ? (void*)st : contactForce, S->dfc, vb, hipMemcpyDeviceToHost, s), "d2h f");
  const int rc2 = c->hip(hipStreamSynchronize(s), "sync");
  if (rc || rc2) return rc ? rc : rc2;
  if (st) std::memcpy(contactForce, st, vb);
  for (long long q = 0; q < 3ll * N; q++)
    if (!std::isfinite(contactForce[q]))
      return c->fail(PDG_E_NONFINITE, "NaN returned by contact force evaluation");
  return PDG_OK;
}

int pdg_contact_force_density(pdg_ctx* h, double* contactForce) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  if (!c || (c->N > 0 && !contactForce)) return PDG_E_ARG;
  if (!c->contact) return c->fail(PDG_E_ARG, "no contact model (pdg_set_contact)");
  (void)hipSetDevice(c->device);
  return c->download_vec3(c->contact->fc, contactForce);
}

}  // extern "C"
