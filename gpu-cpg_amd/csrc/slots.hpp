// Room on the device for the level and scheduled loops of every handle,
// batch, server and no-allocation call of the process.
//
// A wave of such a loop waits for other waves of the same loop, so a loop in
// flight needs all its blocks resident: loops each of which is half
// dispatched, on a device that the others fill, would wait until their spin
// limits.  One loop's grid is kept below that by itself (resident_blocks);
// this counts the blocks of all loops in flight.  A loop alone gets the grid
// it asks for.  Beside others it gets at most half of what is left (all but
// 256 slots where that is more), and where nothing is left one block, which
// is resident whenever it runs; so nothing waits here.
#pragma once
#include <algorithm>
#include <mutex>

namespace cpg {

class LoopSlots {
 public:
  // The current device's (sfxt.hip, which knows how many blocks it holds).
  static LoopSlots& current();

  void set_capacity(int blocks) { capacity_ = blocks; }
  // Slots for a loop of up to `want` blocks, at least `least`; a block takes
  // `per_block` slots (one held to an XCD takes that XCD's share of all
  // eight).  Returns the blocks granted.
  int take(int want, int per_block, int least, int* slots) {
    std::lock_guard<std::mutex> lk(mu_);
    int blocks = std::max(want, least);
    if (used_ > 0) {
      const int left = capacity_ - used_;
      blocks = std::max(least, std::min(want, std::max(left / 2, left - 256) / per_block));
    }
    *slots = blocks * per_block;
    used_ += *slots;
    return blocks;
  }
  void give(int slots) {
    std::lock_guard<std::mutex> lk(mu_);
    used_ -= slots;
  }

 private:
  std::mutex mu_;
  int capacity_ = 0;
  int used_ = 0;
};

// The slots of one loop in flight.
class LoopLease {
 public:
  LoopLease() = default;
  LoopLease(const LoopLease&) = delete;
  LoopLease& operator=(const LoopLease&) = delete;
  ~LoopLease() { release(); }
  int take(int want, int per_block = 1, int least = 1) {
    release();
    from_ = &LoopSlots::current();
    return from_->take(want, per_block, least, &slots_);
  }
  // Once the loop has ended.
  void release() {
    if (from_) from_->give(slots_);
    from_ = nullptr;
  }

 private:
  LoopSlots* from_ = nullptr;
  int slots_ = 0;
};

}  // namespace cpg
