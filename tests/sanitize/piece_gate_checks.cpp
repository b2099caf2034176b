// PieceGate: every thread sees every piece once it is raised, a failure ends
// all waits, and a thread that waits long takes no processor time.
#include <sys/resource.h>

#include <cstdio>
#include <limits>
#include <vector>

#include "piece_gate.h"

static double thread_seconds() {
  rusage u;
  getrusage(RUSAGE_THREAD, &u);
  return u.ru_utime.tv_sec + u.ru_stime.tv_sec + 1e-6 * (u.ru_utime.tv_usec + u.ru_stime.tv_usec);
}

int main() {
  constexpr int kThreads = 4, kPieces = 2000;
  int bad = 0;
  for (int late : {0, 1}) {
    mdx::PieceGate gate;
    std::vector<int> data(kPieces, 0);
    std::vector<long> sum(kThreads, 0);
    std::vector<double> used(kThreads, 0.0);
    std::vector<std::thread> pool;
    for (int t = 0; t < kThreads; t++)
      pool.emplace_back([&, t] {
        const double before = thread_seconds();
        for (int k = 0; k < kPieces; k++) {
          if (gate.wait(k) == std::numeric_limits<int>::max()) return;
          if (k == 0) used[t] = thread_seconds() - before;
          sum[t] += data[k];
        }
      });
    if (late) std::this_thread::sleep_for(std::chrono::milliseconds(400));
    for (int k = 0; k < kPieces; k++) {
      data[k] = k + 1;
      gate.raise(k + 1);
    }
    for (auto &th : pool) th.join();
    for (int t = 0; t < kThreads; t++) {
      if (sum[t] != (long)kPieces * (kPieces + 1) / 2) bad++;
      if (late && used[t] > 0.1) {
        std::printf("%.0f ms of processor time in a wait of 400 ms\n", 1e3 * used[t]);
        bad++;
      }
    }
  }
  mdx::PieceGate gate;
  std::vector<std::thread> pool;
  std::atomic<int> ended{0};
  for (int t = 0; t < kThreads; t++)
    pool.emplace_back([&] {
      for (int k = 0; gate.wait(k) != std::numeric_limits<int>::max(); k++) {
      }
      ended++;
    });
  gate.raise(1);
  gate.raise(std::numeric_limits<int>::max());
  for (auto &th : pool) th.join();
  if (ended != kThreads) bad++;
  std::printf("%d faults\n", bad);
  return bad ? 1 : 0;
}
