// Small result buffers that calls share instead of allocating.  Host code only.
#pragma once
#include <mutex>

namespace azb {

// Which of a fixed set of slots are taken.
class SlotSet {
 public:
  static constexpr int kSlots = 16;
  // a free slot's number, or -1
  int take() {
    std::lock_guard<std::mutex> lock(mu_);
    for (int i = 0; i < kSlots; ++i)
      if (!(taken_ >> i & 1)) {
        taken_ |= 1u << i;
        return i;
      }
    return -1;
  }
  void give(int i) {
    std::lock_guard<std::mutex> lock(mu_);
    taken_ &= ~(1u << i);
  }

 private:
  std::mutex mu_;
  unsigned taken_ = 0;
};

// One call's hold on a slot.  From the first queued work that touches the slot until a
// successful wait() the slot must not go to another call, so a call that returns early
// waits here, and where even that fails (the stream is being captured, the device is
// lost) the slot stays taken for good: later calls find another or allocate.
// Wait: callable, 0 once everything queued so far has ended.
template <class Wait>
class SlotLease {
 public:
  explicit SlotLease(Wait wait) : wait_(wait) {}
  SlotLease(const SlotLease&) = delete;
  SlotLease& operator=(const SlotLease&) = delete;
  ~SlotLease() {
    if (index_ >= 0 && (!queued_ || wait_() == 0)) set_->give(index_);
  }
  // the slot's number, or -1 when all are taken
  int take(SlotSet& set) {
    set_ = &set;
    return index_ = set.take();
  }
  void queued() { queued_ = true; }
  int wait() {
    const int rc = wait_();
    if (rc == 0) queued_ = false;
    return rc;
  }

 private:
  Wait wait_;
  SlotSet* set_ = nullptr;
  int index_ = -1;
  bool queued_ = false;
};

}  // namespace azb
