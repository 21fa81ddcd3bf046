// Sharing the GPU between sweeps: a budget for the threads of this process, and
// when to try again after others were in the way.
#pragma once
#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace sa {

// Units of a resource that host threads share, handed out in the order in
// which the threads ask, so that a large demand is not passed over by small
// ones.
class Budget {
 public:
  explicit Budget(int total) : total_(total) {}

  // Waits for its turn and the units; false at once when there are not that
  // many in all.
  bool take(int units) {
    if (units > total_) return false;
    std::unique_lock<std::mutex> lk(mu_);
    const uint64_t mine = asked_++;
    cv_.wait(lk, [&] { return mine == served_ && used_ + units <= total_; });
    served_++;
    used_ += units;
    lk.unlock();
    cv_.notify_all();      // the next in line may fit beside this one
    return true;
  }
  void give(int units) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      used_ -= units;
    }
    cv_.notify_all();
  }

 private:
  const int total_;
  int used_ = 0;
  uint64_t asked_ = 0, served_ = 0;
  std::mutex mu_;
  std::condition_variable cv_;
};

// After f failures in a row the next 2^(f-1) - 1 turns, 255 at most, pass without
// a try: one failure costs nothing more, a lasting cause one try in 256 turns.
class Backoff {
 public:
  bool due() {
    if (rest_ == 0) return true;
    rest_--;
    return false;
  }
  void succeeded() { failures_ = 0; }
  void failed() {
    failures_ = std::min(failures_ + 1, 9);
    rest_ = (1 << (failures_ - 1)) - 1;
  }

 private:
  int failures_ = 0, rest_ = 0;
};

}  // namespace sa
