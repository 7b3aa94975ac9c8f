// When a conjugate-gradient solve ends, and how (cg_ends and cg_broke_down of
// peridigm_amd/csrc/pdg_qs_status.hpp), against the host loop that the device's
// decision stands for: it takes an iteration, looks at the residual and the
// breakdowns of the iterations before it, and only then notes that this one
// had p.Kp <= 0. Every pair of an iteration that breaks down (and all later
// ones) and one from which the residual is within the tolerance, with every
// limit.
#include <cstdio>

#include "../../peridigm_amd/csrc/pdg_qs_status.hpp"

enum { CONVERGED, NOT_CONVERGED, BROKE_DOWN };

int main() {
  struct { int maxit; double bnorm, tol; } c{0, 2.0, 1e-3};
  auto rr = [&](int it, int from) { return it >= from ? 0.0 : 4.0; };  // squared residual
  int bad = 0, cases = 0;
  for (int maxit = 0; maxit <= 26; maxit++)
    for (int broken = 1; broken <= 30; broken++)
      for (int from = 0; from <= 30; from++, cases++) {
        c.maxit = maxit;
        // the host loop
        int want = -1, it = 0, brk = 0;
        if (rr(0, from) == 0.0) want = CONVERGED;
        while (want < 0 && it < maxit) {
          it++;
          if (it <= 8 || it % 4 == 0 || it == maxit) {
            if (brk) { want = BROKE_DOWN; break; }
            if (rr(it, from) == 0.0) { want = CONVERGED; break; }
          }
          if (it >= broken) brk = 1;
        }
        if (want < 0) want = brk ? BROKE_DOWN : NOT_CONVERGED;
        // the device
        int k = 0, b = 0;
        while (!pdg::cg_ends(&c, k, b, rr(k, from))) {
          k++;
          if (k >= broken) b = 1;
        }
        const int got = pdg::cg_broke_down(&c, k, b, rr(k, from)) ? BROKE_DOWN
                        : rr(k, from) == 0.0                                     ? CONVERGED
                                                                                 : NOT_CONVERGED;
        if (got != want && bad++ < 10)
          std::printf("limit %d, breakdown at %d, converged from %d: %d, not %d\n", maxit, broken,
                      from, got, want);
      }
  std::printf("%d cases, %d wrong\n", cases, bad);
  return bad != 0;
}
