// glx_slots.h -- the blocks that solves in flight keep resident on a device:
// plain C++, so that it can be tested without one.
#pragma once

#include <condition_variable>
#include <mutex>

namespace glx {

// The slots a launch of resident blocks takes: workgroups go round the eight
// XCDs in turn, so an XCD holds up to ceil(blocks / 8) of them.  Counted in
// whole rounds, launches that fit the device fit every XCD; counted by blocks,
// 65 and 190 blocks (255 of 256 CUs) could want 9 + 24 of one XCD's 32, and two
// launches that each miss a block on another XCD would wait for each other
// until their polls run out.
constexpr int kXcds = 8;
constexpr int resident_slots(int blocks) { return (blocks + kXcds - 1) / kXcds * kXcds; }

// A count that callers take from and give back, first come first served: one
// that asks for much is not passed over for ever by others that fit beside
// what is in use.
class FairSlots {
 public:
  // Waits until every earlier caller has its slots and n more are within cap.
  void acquire(int n, int cap) {
    std::unique_lock<std::mutex> l(mu_);
    const unsigned long mine = next_++;
    cv_.wait(l, [&] { return serving_ == mine && (used_ + n <= cap || used_ == 0); });
    serving_++;
    used_ += n;
    cv_.notify_all();
  }
  void release(int n) {
    {
      std::lock_guard<std::mutex> l(mu_);
      used_ -= n;
    }
    cv_.notify_all();
  }
  // slots in use, and callers waiting
  int used() {
    std::lock_guard<std::mutex> l(mu_);
    return used_;
  }
  int waiting() {
    std::lock_guard<std::mutex> l(mu_);
    return int(next_ - serving_);
  }

 private:
  std::mutex mu_;
  std::condition_variable cv_;
  unsigned long next_ = 0, serving_ = 0;
  int used_ = 0;
};

}  // namespace glx
