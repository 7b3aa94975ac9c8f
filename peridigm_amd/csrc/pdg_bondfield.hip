// Bond fields across the boundary: Bond_Damage, FP64 in list order on the host
// and one bit a bond in the internal rows on the device.
//
// A field of zeros and ones goes up in chunks, each packed into bits in list
// order as it arrives; one kernel then gathers the internal rows' words from
// those bits through the bond index map, and one checks that both ends of
// every bond agree. Coming back, the broken bonds' bits are set in list order
// (few, so atomics are cheap) and the host threads only widen bits to doubles,
// front to back. A host that gathers and scatters single bonds through the
// index maps took 5 to 8 ms a call for 3M bonds; here the copy over PCIe, 24
// MB at 30 GB/s, and the caller's pages bound it: 3.1M bonds 1.0 ms up and
// 0.9 ms down.

#include <algorithm>
#include <cstring>

#include "pdg_ctx.hpp"

namespace pdg {
namespace {

constexpr long long kChunk = 1ll << 22;  // doubles (32 MB), a multiple of 64

inline unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

// Bits of n field values in list order (a wave per word); bad[0] is set by a
// value that is neither 0 nor 1.
__global__ __launch_bounds__(256) void k_pack_bits(long long n, const double* __restrict__ bd,
                                                   unsigned long long* __restrict__ bits,
                                                   int* __restrict__ bad) {
  const long long b = (long long)blockIdx.x * 256 + threadIdx.x;
  const double d = b < n ? bd[b] : 0.0;
  const unsigned long long m = __ballot(d == 1.0);
  const bool wrong = __ballot(d != 0.0 && d != 1.0) != 0ull;
  if ((threadIdx.x & 63) == 0 && b < n) {
    bits[b >> 6] = m;
    if (wrong) bad[0] = 1;
  }
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

// bad[1] is set by a bond that only one end has broken: a wave per node.
__global__ __launch_bounds__(256) void k_check_ends(int n, const int* __restrict__ row,
                                                    const int* __restrict__ mw,
                                                    const int* __restrict__ col,
                                                    const int* __restrict__ rev,
                                                    const unsigned long long* __restrict__ words,
                                                    int* __restrict__ bad) {
  const long long t = wave_index();
  if (t >= n) return;
  const int i = (int)t, lane = threadIdx.x & 63;
  const int rs = row[i], deg = row[i + 1] - rs, w0 = mw[i];
  bool wrong = false;
  for (int k = lane; k < deg; k += 64) {
    const int j = col[rs + k], r = rev[rs + k] - row[j];
    const unsigned long long a = words[w0 + (k >> 6)] >> (k & 63);
    const unsigned long long b = words[mw[j] + (r >> 6)] >> (r & 63);
    wrong |= ((a ^ b) & 1ull) != 0ull;
  }
  if (__ballot(wrong) && lane == 0) bad[1] = 1;
}

// The checked words become the mask (an accepted field only).
__global__ __launch_bounds__(256) void k_take_words(long long n, const unsigned long long* __restrict__ words,
                                                    const int* __restrict__ bad,
                                                    unsigned long long* __restrict__ mask) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t < n && !bad[0] && !bad[1]) mask[t] = words[t];
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
  void* p[] = {d_src, d_rev, d_lbits, d_words, d_chunk, d_bad};
  for (void* q : p) if (q) (void)hipFree(q);
  d_src = d_rev = d_bad = nullptr;
  d_lbits = d_words = nullptr;
  d_chunk = nullptr;
}

int Ctx::bond_maps(bool reverse) {
  auto A = [&](void** p, size_t bytes) { return hip(hipMalloc(p, std::max<size_t>(bytes, 64)), "alloc bond maps"); };
  const size_t nb = (size_t)B;
  int rc = PDG_OK;
  if (!d_bad) {
    rc = A((void**)&d_src, 4 * nb);
    if (!rc) rc = A((void**)&d_lbits, 8 * ((nb + 63) / 64));
    if (!rc) rc = A((void**)&d_words, 8 * (size_t)mw.back());
    if (!rc) rc = A((void**)&d_chunk, 8 * (size_t)std::min<long long>(B, kChunk));
    if (!rc) rc = A((void**)&d_bad, 8);
    if (!rc && nb) rc = hip(hipMemcpyAsync(d_src, src.data(), 4 * nb, hipMemcpyHostToDevice, stream), "h2d bond map");
    if (rc) { free_bond_maps(); return rc; }
  }
  if (reverse && !d_rev) {
    rc = A((void**)&d_rev, 4 * nb);
    if (!rc && nb) rc = hip(hipMemcpyAsync(d_rev, rev.data(), 4 * nb, hipMemcpyHostToDevice, stream), "h2d bond map");
  }
  return rc;
}

// Host field (list order) -> mask words. A rejected field leaves the mask as
// it was.
int Ctx::upload_mask(const double* bd, bool check_symmetric) {
  const long long nw = mw.back();
  if (!bd)  // no field: every bond intact
    return hip(hipMemsetAsync(d_mask, 0, (size_t)nw * 8, stream), "zero mask");
  if (B == 0) return PDG_OK;
  int rc = bond_maps(check_symmetric);
  if (rc) return rc;
  hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(256), 0, stream, 1ll, (unsigned long long*)d_bad);
  for (long long b = 0; b < B; b += kChunk) {
    const long long n = std::min(kChunk, B - b);
    rc = hip(hipMemcpyAsync(d_chunk, bd + b, 8 * (size_t)n, hipMemcpyHostToDevice, stream), "h2d bond field");
    if (rc) return rc;
    hipLaunchKernelGGL(k_pack_bits, dim3(blocks_for(n)), dim3(256), 0, stream, n, d_chunk,
                       d_lbits + b / 64, d_bad);
  }
  const dim3 per_node = wave_grid(N);
  hipLaunchKernelGGL(k_rows_from_bits, per_node, dim3(256), 0, stream, N, d_row, d_mw, d_src,
                     d_lbits, d_words);
  if (check_symmetric)
    hipLaunchKernelGGL(k_check_ends, per_node, dim3(256), 0, stream, N, d_row, d_mw, d_col, d_rev,
                       d_words, d_bad);
  hipLaunchKernelGGL(k_take_words, dim3(blocks_for(nw)), dim3(256), 0, stream, nw, d_words, d_bad, d_mask);
  rc = hip(hipGetLastError(), "bond field");
  int bad[2] = {0, 0};
  if (!rc) rc = hip(hipMemcpyAsync(bad, d_bad, 8, hipMemcpyDeviceToHost, stream), "d2h");
  const int rc2 = hip(hipStreamSynchronize(stream), "sync");
  if (rc || rc2) return rc ? rc : rc2;
  if (bad[0]) return fail(PDG_E_UNSUPPORTED, "bond damage values must be 0 or 1");
  if (bad[1]) return fail(PDG_E_UNSUPPORTED, "bond damage must be symmetric (d_ij == d_ji)");
  return PDG_OK;
}

int Ctx::download_mask(double* bd) {
  if (B == 0) return hip(hipStreamSynchronize(stream), "sync");
  int rc = bond_maps(false);
  if (rc) return rc;
  const long long nw = (B + 63) / 64;
  hipLaunchKernelGGL(k_zero_words, dim3(blocks_for(nw)), dim3(256), 0, stream, nw, d_lbits);
  hipLaunchKernelGGL(k_bits_from_rows, wave_grid(N), dim3(256), 0, stream, N,
                     d_row, d_mw, d_src, d_mask, d_lbits);
  rc = hip(hipGetLastError(), "bond field");
  if (rc) return rc;
  std::vector<unsigned long long> own;
  unsigned long long* w = reinterpret_cast<unsigned long long*>(stage(8 * (size_t)nw));
  if (!w) {
    own.resize(nw);
    w = own.data();
  }
  rc = hip(hipMemcpyAsync(w, d_lbits, 8 * (size_t)nw, hipMemcpyDeviceToHost, stream), "d2h bond bits");
  if (!rc) rc = hip(hipStreamSynchronize(stream), "sync");
  if (rc) return rc;
  const unsigned nt = B < (1ll << 18) ? 1 : B < (1ll << 22) ? 4 : 8;
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
