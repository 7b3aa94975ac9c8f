// Bond fields across the boundary: Bond_Damage, FP64 in list order on the host
// and one bit a bond in the internal rows on the device.
//
// Host threads pack a field of zeros and ones into bits in list order, front to
// back, and a 64th of it goes up; one kernel then gathers the internal rows'
// words from those bits through the bond index map, and one checks the other
// end of every broken bond. Coming back, the broken bonds' bits are set in list
// order (few, so atomics are cheap) and the host threads only widen bits to
// doubles, front to back. Bound by host memory: the field is read once.
// The whole field over PCIe, packed by a kernel, was bound by the copy from
// pageable memory, host threads that gather single bonds through the map by
// those. Drop-in force with a field, 640,000 nodes, 55M bonds, none, a fifth and
// all of them broken: gather 13.4, 19.1, 15.9 ms, whole field 16.1 in each, now
// 4.1, 5.2, 8.2; 980 nodes: 196, 307, 233 us, 355 (130 repeated), now 82, 92, 118.

#include <emmintrin.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstring>

#include "pdg_ctx.hpp"

namespace pdg {
namespace {

inline unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

// Threads that pack or widen a field of nb bonds (starting one takes as long as
// a core takes for some 50,000 bonds).
inline unsigned field_threads(long long nb) { return nb < (1ll << 18) ? 1 : nb < (1ll << 22) ? 4 : 8; }

// Bits of m <= 64 field values; `wrong` is set by a value other than 0 and 1.
// Whole words with SSE2, 21 ns each on one core whatever they hold (a value at a
// time takes 64 to 75).
inline unsigned long long pack_bits(const double* v, int m, bool& wrong) {
  unsigned long long bits = 0ull;
  if (m < 64) {
    for (int k = 0; k < m; k++) {
      wrong |= v[k] != 0.0 && v[k] != 1.0;
      bits |= (unsigned long long)(v[k] == 1.0) << k;
    }
    return bits;
  }
  const __m128d one = _mm_set1_pd(1.0), zero = _mm_setzero_pd();
  __m128d ok = _mm_cmpeq_pd(zero, zero);
  for (int k = 0; k < 64; k += 16) {
    __m128i c[8];  // two comparisons each, 16 values
    for (int q = 0; q < 8; q++) {
      const __m128d x = _mm_loadu_pd(v + k + 2 * q), o = _mm_cmpeq_pd(x, one);
      ok = _mm_and_pd(ok, _mm_or_pd(o, _mm_cmpeq_pd(x, zero)));
      c[q] = _mm_castpd_si128(o);
    }
    // narrowed to a byte each
    for (int q = 0; q < 8; q += 2) c[q] = _mm_packs_epi32(c[q], c[q + 1]);
    c[0] = _mm_packs_epi32(c[0], c[2]);
    c[4] = _mm_packs_epi32(c[4], c[6]);
    bits |= (unsigned long long)(unsigned)_mm_movemask_epi8(_mm_packs_epi16(c[0], c[4])) << k;
  }
  wrong |= _mm_movemask_pd(ok) != 3;
  return bits;
}

// List-order index of every internal bond where the list's rows ascend and
// have at most 128 entries: the row's first index plus the number of smaller
// ids in the row. A wave per node. (Computed, the map is there in 0.2 ms at 55M
// bonds; the copy of the host's took 8.)
__global__ __launch_bounds__(256) void k_src_by_rank(int n, const int* __restrict__ row,
                                                     const int* __restrict__ col,
                                                     const int* __restrict__ perm,
                                                     const int* __restrict__ first,
                                                     int* __restrict__ src) {
  const long long t = wave_index();
  if (t >= n) return;
  const int i = (int)t, lane = threadIdx.x & 63;
  const int rs = row[i], deg = row[i + 1] - rs;
  const int a = lane < deg ? perm[col[rs + lane]] : INT_MAX;
  const int b = lane + 64 < deg ? perm[col[rs + lane + 64]] : INT_MAX;
  int ra = 0, rb = 0;
  for (int k = 0; k < min(deg, 64); k++) {
    const int v = __shfl(a, k);
    ra += v < a;
    rb += v < b;
  }
  for (int k = 0; k < deg - 64; k++) {
    const int v = __shfl(b, k);
    ra += v < a;
    rb += v < b;
  }
  if (lane < deg) src[rs + lane] = first[i] + ra;
  if (lane + 64 < deg) src[rs + lane + 64] = first[i] + rb;
}

// Mask words of the internal rows from the list-order bits: a wave per node.
__global__ __launch_bounds__(256) void k_rows_from_bits(int n, const int* __restrict__ row,
                                                        const int* __restrict__ mw,
                                                        const int* __restrict__ src,
                                                        const unsigned long long* __restrict__ bits,
                                                        unsigned long long* __restrict__ words) {
  const long long t = wave_index();
  if (t >= n) return;
  const int i = (int)t, lane = threadIdx.x & 63;
  const int rs = row[i], deg = row[i + 1] - rs, w0 = mw[i];
  for (int k0 = 0; k0 < deg; k0 += 64) {
    bool broken = false;
    if (k0 + lane < deg) {
      const unsigned s = (unsigned)src[rs + k0 + lane];
      broken = (bits[s >> 6] >> (s & 63)) & 1ull;
    }
    const unsigned long long m = __ballot(broken);
    if (lane == 0) words[w0 + (k0 >> 6)] = m;
  }
}

// *bad is set by a broken bond whose other end is intact: a wave per node, which
// looks the node up in the other end's row for each of its broken bonds, four
// rows in flight.
__global__ __launch_bounds__(256) void k_check_ends(int n, const int* __restrict__ row,
                                                    const int* __restrict__ mw,
                                                    const int* __restrict__ col,
                                                    const unsigned long long* __restrict__ words,
                                                    int* __restrict__ bad) {
  constexpr int U = 4;
  const long long t = wave_index();
  if (t >= n) return;
  const int i = (int)t, lane = threadIdx.x & 63;
  const int rs = row[i], deg = row[i + 1] - rs, w0 = mw[i];
  bool wrong = false;
  for (int k0 = 0; k0 < deg; k0 += 64) {
    unsigned long long m = words[w0 + (k0 >> 6)];
    if (m == 0ull) continue;
    int rj = 0, dj = 0, wj = 0;  // lane k's bond's other end
    if (k0 + lane < deg) {
      const int j = col[rs + k0 + lane];
      rj = row[j];
      dj = row[j + 1] - rj;
      wj = mw[j];
    }
    while (m != 0ull) {
      int d[U], w[U], c0[U], c1[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int b = m != 0ull ? __ffsll(m) - 1 : 0;  // past the last: no row
        const int r = __shfl(rj, b);
        d[u] = m != 0ull ? __shfl(dj, b) : 0;
        w[u] = __shfl(wj, b);
        m &= m - 1ull;
        c0[u] = lane < d[u] ? col[r + lane] : -1;
        c1[u] = lane + 64 < d[u] ? col[r + lane + 64] : -1;
        for (int q = lane + 128; q < d[u]; q += 64)
          if (col[r + q] == i) wrong = wrong || !((words[w[u] + (q >> 6)] >> (q & 63)) & 1ull);
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (c0[u] == i) wrong = wrong || !((words[w[u]] >> lane) & 1ull);
        if (c1[u] == i) wrong = wrong || !((words[w[u] + 1] >> lane) & 1ull);
      }
    }
  }
  if (__ballot(wrong) && lane == 0) *bad = 1;
}

// The checked words become the mask (an accepted field only).
__global__ __launch_bounds__(256) void k_take_words(long long n, const unsigned long long* __restrict__ words,
                                                    const int* __restrict__ bad,
                                                    unsigned long long* __restrict__ mask) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t < n && !*bad) mask[t] = words[t];
}

__global__ __launch_bounds__(256) void k_zero_words(long long n, unsigned long long* __restrict__ w) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t < n) w[t] = 0ull;
}

// List-order bits of the broken bonds (cleared before): a wave per node.
__global__ __launch_bounds__(256) void k_bits_from_rows(int n, const int* __restrict__ row,
                                                        const int* __restrict__ mw,
                                                        const int* __restrict__ src,
                                                        const unsigned long long* __restrict__ mask,
                                                        unsigned long long* __restrict__ bits) {
  const long long t = wave_index();
  if (t >= n) return;
  const int i = (int)t, lane = threadIdx.x & 63;
  const int rs = row[i], deg = row[i + 1] - rs, w0 = mw[i];
  for (int k0 = 0; k0 < deg; k0 += 64) {
    const unsigned long long w = mask[w0 + (k0 >> 6)];
    if (w == 0ull) continue;
    if (k0 + lane < deg && ((w >> lane) & 1ull)) {
      const unsigned s = (unsigned)src[rs + k0 + lane];
      atomicOr(&bits[s >> 6], 1ull << (s & 63));
    }
  }
}

}  // namespace

void Ctx::free_bond_maps() {
  if (d_src) (void)hipFree(d_src);
  d_src = d_bad = nullptr;
  d_lbits = d_words = nullptr;
}

// Device memory of the fields and the bond index map. `first` is a place in
// memory that copies may read until the stream is synchronised (n ints).
int Ctx::bond_maps(int* first) {
  if (d_src) return PDG_OK;
  auto up = [](size_t bytes) { return (bytes + 63) & ~(size_t)63; };
  const size_t sb = up(4 * (size_t)B), wb = up(8 * (size_t)mw.back()), lw = ((size_t)B + 63) / 64;
  char* p = nullptr;
  int rc = hip(hipMalloc((void**)&p, sb + wb + 8 * (lw + 1)), "alloc bond maps");
  if (rc) {
    (void)hipGetLastError();
    return rc;
  }
  d_src = reinterpret_cast<int*>(p);
  d_words = reinterpret_cast<unsigned long long*>(p + sb);
  d_lbits = reinterpret_cast<unsigned long long*>(p + sb + wb);
  d_bad = reinterpret_cast<int*>(d_lbits + lw);  // cleared with the bits' copy
  if (list_ascends && ntiles > 0) {
    for (int k = 0; k < N; k++) first[k] = (int)(head[perm[k]] - perm[k]);
    int* const d_first = reinterpret_cast<int*>(d_y);
    rc = hip(hipMemcpyAsync(d_first, first, 4 * (size_t)N, hipMemcpyHostToDevice, stream), "h2d rows");
    if (!rc)
      hipLaunchKernelGGL(k_src_by_rank, wave_grid(N), dim3(256), 0, stream, N, d_row, d_col, d_perm,
                         d_first, d_src);
  } else {
    rc = hip(hipMemcpyAsync(d_src, src.data(), 4 * (size_t)B, hipMemcpyHostToDevice, stream), "h2d bond map");
  }
  if (rc) {
    (void)hipStreamSynchronize(stream);
    free_bond_maps();
  }
  return rc;
}

// Host field (list order) -> mask words. A rejected field leaves the mask as
// it was.
int Ctx::upload_mask(const double* bd, bool check_symmetric) {
  const long long nw = mw.back(), lw = (B + 63) / 64;
  if (!bd)  // no field: every bond intact
    return hip(hipMemsetAsync(d_mask, 0, (size_t)nw * 8, stream), "zero mask");
  if (B == 0) return PDG_OK;
  // bits and rows behind the place of a small mesh's positions, which may be
  // on their way
  const size_t at = N <= kHostOrderMax ? (24 * (size_t)N + 63) & ~(size_t)63 : 0;
  const size_t bytes = 8 * (size_t)(lw + 1) + 4 * (size_t)N + 8;
  std::vector<char> own;
  char* st = stage(at + bytes);
  if (st) {
    st += at;
  } else {
    own.resize(bytes);
    st = own.data();
  }
  unsigned long long* const w = reinterpret_cast<unsigned long long*>(st);
  int* const first = reinterpret_cast<int*>(w + lw + 1);
  int* const bad = first + N;
  w[lw] = 0ull;
  std::atomic<bool> wrong{false};
  const unsigned nt = field_threads(B);
  on_threads(nt, [&](unsigned t) {
    bool bad_value = false;
    for (long long q = lw * t / nt; q < lw * (t + 1) / nt; q++)
      w[q] = pack_bits(bd + 64 * q, (int)std::min<long long>(64, B - 64 * q), bad_value);
    if (bad_value) wrong = true;
  });
  if (wrong) return fail(PDG_E_UNSUPPORTED, "bond damage values must be 0 or 1");
  int rc = bond_maps(first);
  if (rc) return rc;
  rc = hip(hipMemcpyAsync(d_lbits, w, 8 * (size_t)(lw + 1), hipMemcpyHostToDevice, stream), "h2d bond bits");
  hipLaunchKernelGGL(k_rows_from_bits, wave_grid(N), dim3(256), 0, stream, N, d_row, d_mw, d_src,
                     d_lbits, d_words);
  if (check_symmetric)
    hipLaunchKernelGGL(k_check_ends, wave_grid(N), dim3(256), 0, stream, N, d_row, d_mw, d_col,
                       d_words, d_bad);
  hipLaunchKernelGGL(k_take_words, dim3(blocks_for(nw)), dim3(256), 0, stream, nw, d_words, d_bad, d_mask);
  if (!rc) rc = hip(hipGetLastError(), "bond field");
  *bad = 0;
  if (!rc && check_symmetric)
    rc = hip(hipMemcpyAsync(bad, d_bad, 4, hipMemcpyDeviceToHost, stream), "d2h");
  const int rc2 = hip(hipStreamSynchronize(stream), "sync");
  if (rc || rc2) return rc ? rc : rc2;
  return *bad ? fail(PDG_E_UNSUPPORTED, "bond damage must be symmetric (d_ij == d_ji)") : PDG_OK;
}

int Ctx::download_mask(double* bd) {
  if (B == 0) return hip(hipStreamSynchronize(stream), "sync");
  const long long nw = (B + 63) / 64;
  std::vector<char> own;
  char* st = stage(8 * (size_t)nw + 4 * (size_t)N);
  if (!st) {
    own.resize(8 * (size_t)nw + 4 * (size_t)N);
    st = own.data();
  }
  unsigned long long* const w = reinterpret_cast<unsigned long long*>(st);
  int rc = bond_maps(reinterpret_cast<int*>(st + 8 * nw));
  if (rc) return rc;
  hipLaunchKernelGGL(k_zero_words, dim3(blocks_for(nw)), dim3(256), 0, stream, nw, d_lbits);
  hipLaunchKernelGGL(k_bits_from_rows, wave_grid(N), dim3(256), 0, stream, N,
                     d_row, d_mw, d_src, d_mask, d_lbits);
  rc = hip(hipGetLastError(), "bond field");
  if (rc) return rc;
  rc = hip(hipMemcpyAsync(w, d_lbits, 8 * (size_t)nw, hipMemcpyDeviceToHost, stream), "d2h bond bits");
  if (!rc) rc = hip(hipStreamSynchronize(stream), "sync");
  if (rc) return rc;
  const unsigned nt = field_threads(B);
  on_threads(nt, [&](unsigned t) {
    for (long long q = nw * t / nt; q < nw * (t + 1) / nt; q++) {
      double* out = bd + 64 * q;
      const int m = (int)std::min<long long>(64, B - 64 * q);
      if (w[q] == 0ull) {
        std::memset(out, 0, 8 * (size_t)m);
      } else {
        for (int k = 0; k < m; k++) out[k] = (double)((w[q] >> k) & 1ull);
      }
    }
  });
  return PDG_OK;
}

}  // namespace pdg
