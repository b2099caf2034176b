// piece_gate.h - how helper threads wait for pieces of a transfer.
#pragma once
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>

namespace mdx {

// A count of pieces that are ready, raised by one thread and waited for by
// others.  Between two pieces of a running transfer the wait is shorter than a
// wake-up, so a waiting thread yields for kSpin first; then it sleeps, as the
// first piece may lie behind milliseconds of GPU work and the cores belong to
// other ranks of the host meanwhile.
class PieceGate {
 public:
  void raise(int count) {
    {
      std::lock_guard<std::mutex> lock(m_);
      ready_.store(count, std::memory_order_release);
    }
    cv_.notify_all();
  }
  // the count, once it is above `piece`
  int wait(int piece) {
    const auto until = std::chrono::steady_clock::now() + kSpin;
    for (;;) {
      const int r = ready_.load(std::memory_order_acquire);
      if (r > piece) return r;
      if (std::chrono::steady_clock::now() >= until) break;
      std::this_thread::yield();
    }
    std::unique_lock<std::mutex> lock(m_);
    cv_.wait(lock, [&] { return ready_.load(std::memory_order_relaxed) > piece; });
    return ready_.load(std::memory_order_relaxed);
  }

 private:
  static constexpr std::chrono::microseconds kSpin{50};
  std::atomic<int> ready_{0};
  std::mutex m_;
  std::condition_variable cv_;
};

}  // namespace mdx
