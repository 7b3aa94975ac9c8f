// How a conjugate-gradient solve on the device tells the host that it ended
// (host code as well: tests build it without HIP).
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>

#define PDG_BOTH __host__ __device__ inline
#else
#include <cmath>
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

// The end of a solve after `it` iterations with squared residual rr, `brk` set
// when an iteration so far had p.Kp <= 0. The residual is looked at for it up to
// 8, every fourth and the last one (a NaN ends the solve). A solve whose residual
// is found within the tolerance there has converged, also when p.Kp came out as 0
// because nothing was left to correct; otherwise a breakdown ends it.
// S holds maxit, bnorm and tol.
template <class S>
PDG_BOTH bool cg_ends(const S* c, int it, int brk, double rr) {
  const bool look = it <= 8 || it % 4 == 0 || it >= c->maxit;
  return brk || it >= c->maxit || (look && !(sqrt(rr) / c->bnorm > c->tol));
}
template <class S>
PDG_BOTH bool cg_broke_down(const S* c, int it, int brk, double rr) {
  const bool look = it <= 8 || it % 4 == 0 || it >= c->maxit;
  return brk && !(look && !(sqrt(rr) / c->bnorm > c->tol));
}

}  // namespace pdg
