// A solve's status crosses from the thread that ends it to the one that waits
// (peridigm_amd/csrc/pdg_qs_status.hpp), many times over. Built with a thread
// sanitizer, which reports any field that the two do not hand over in order.
#include <atomic>
#include <cstdio>
#include <thread>

#include "../../peridigm_amd/csrc/pdg_qs_status.hpp"

int main() {
  constexpr int kRounds = 20000;
  static pdg::QsCgStatus status;
  std::atomic<int> turn{0};
  std::thread device([&] {
    for (int k = 1; k <= kRounds; k++) {
      while (turn.load() != k) std::this_thread::yield();
      pdg::cg_status_publish(&status, k & 1, k, 0.5 * k);
    }
  });
  int bad = 0;
  for (int k = 1; k <= kRounds; k++) {
    status = pdg::QsCgStatus{};
    turn.store(k);
    while (!pdg::cg_status_ended(&status)) std::this_thread::yield();
    bad += status.brk != (k & 1) || status.it != k || status.rr != 0.5 * k;
  }
  device.join();
  std::printf("%d rounds, %d wrong\n", kRounds, bad);
  return bad != 0;
}
