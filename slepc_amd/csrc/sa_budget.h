// Units of a resource that host threads share, handed out in the order in
// which the threads ask, so that a large demand is not passed over by small
// ones.
#pragma once
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace sa {

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

}  // namespace sa
