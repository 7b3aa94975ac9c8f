// Conjugate-gradient state on the device, shared by the quasi-static sources.
#pragma once

#include "pdg_device.hpp"
#include "pdg_qs_status.hpp"

namespace pdg {

// One solve's scalars in device memory. `it` counts finished iterations,
// `done` is set by the direction kernel that stops the solve (later launches
// then return at once), rz2 holds r.z of the last two iterations by parity,
// rz the current one.
struct QsCg {
  int done, brk, it, maxit;
  double rz, rz2[2], bnorm, tol;
};

// Arguments of the kernel that starts an iteration: the scalars, the partial
// sums of r.z and r.r that the last one left, and the status to write.
struct QsCgStart {
  QsCg* cg;
  const double* rz_part;
  const double* rr_part;
  int nrz, nrr;
  QsCgStatus* status;
};

#ifdef __HIPCC__
namespace dev {

// v plus its value in another lane of the 16-lane row (a DPP control).
template <int CTRL>
__device__ __forceinline__ double dpp_add64(double v) {
  return v + __hiloint2double(dpp_i<CTRL>(__double2hiint(v)), dpp_i<CTRL>(__double2loint(v)));
}

// Sum over aligned groups of G lanes (4, 8, 16, 32 or 64), in every lane: DPP
// adds inside a row of 16, shuffles across rows. Call with all lanes active.
template <int G>
__device__ __forceinline__ double group_sum64(double v) {
  v = dpp_add64<DPP_QXOR1>(v);
  v = dpp_add64<DPP_QXOR2>(v);
  if (G >= 8) v = dpp_add64<DPP_HMIRROR>(v);
  if (G >= 16) v = dpp_add64<DPP_MIRROR>(v);
  if (G >= 32) v += __shfl_xor(v, 16);
  if (G >= 64) v += __shfl_xor(v, 32);
  return v;
}
__device__ __forceinline__ double wave_sum64(double v) { return group_sum64<64>(v); }

// Sums of two values over a workgroup of T threads, in every thread; sh holds
// 2 T / 64 values. Every thread of the workgroup calls it.
template <int T>
__device__ __forceinline__ void block_sum2(double& a, double& b, double* sh) {
  a = wave_sum64(a);
  b = wave_sum64(b);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    sh[2 * w] = a;
    sh[2 * w + 1] = b;
  }
  __syncthreads();
  a = b = 0.0;
#pragma unroll
  for (int k = 0; k < T / 64; k++) {
    a += sh[2 * k];
    b += sh[2 * k + 1];
  }
}

// Start of iteration cg->it + 1: decides whether the solve stops (cg_ends;
// every workgroup alike, from the same sums in the same order) and gives the
// new direction's beta. Workgroup 0 stores what the iteration's other kernels
// and the host read; rz2 alternates by parity, so no workgroup reads what
// another writes.
template <int T>
__device__ __forceinline__ bool cg_start(const QsCgStart& s, double* sh, double& beta) {
  double rz = 0.0, rr = 0.0;
  for (int i = threadIdx.x; i < s.nrz; i += T) rz += s.rz_part[i];
  for (int i = threadIdx.x; i < s.nrr; i += T) rr += s.rr_part[i];
  const int it = s.cg->it, brk = s.cg->brk;
  const double before = s.cg->rz2[(it + 1) & 1];
  block_sum2<T>(rz, rr, sh);
  const bool stop = cg_ends(s.cg, it, brk, rr);
  beta = it > 0 ? rz / before : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (stop) {
      s.cg->done = 1;
      cg_status_publish(s.status, cg_broke_down(s.cg, it, brk, rr), it, rr);
    } else {
      s.cg->rz = rz;
      s.cg->rz2[it & 1] = rz;
    }
  }
  return stop;
}

}  // namespace dev
#endif

}  // namespace pdg
