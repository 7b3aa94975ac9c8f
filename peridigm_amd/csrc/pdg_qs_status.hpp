// How a conjugate-gradient solve on the device tells the host that it ended
// (host code as well: tests build it without HIP).
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define PDG_BOTH __host__ __device__ inline
#else
#define PDG_BOTH inline
#endif

namespace pdg {

// What the host reads of a stopped solve (pinned memory, written by one thread
// of the device while the host may be looking).
struct QsCgStatus {
  int done, brk, it, pad;
  double rr;
};

// `done` is stored last, with release order for the whole system, so whoever
// sees it sees the other fields; the plain stores it replaced had no order
// between them, and a host that saw `done` alone took a solve that broke down
// or ran out of iterations for one that converged with residual 0.
PDG_BOTH void cg_status_publish(QsCgStatus* s, int brk, int it, double rr) {
  s->brk = brk;
  s->it = it;
  s->rr = rr;
  __atomic_store_n(&s->done, 1, __ATOMIC_RELEASE);
}

// Whether the solve has ended; if so, the other fields hold.
PDG_BOTH bool cg_status_ended(const QsCgStatus* s) {
  return __atomic_load_n(&s->done, __ATOMIC_ACQUIRE) != 0;
}

}  // namespace pdg
