// The shared result slots on the CPU, with a wait that succeeds or fails on request.
#include "../../azeban_amd/csrc/azb_slots.hpp"

#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

using azb::SlotLease;
using azb::SlotSet;

static int waits = 0, wait_rc = 0;
struct Wait {
  int operator()() const {
    ++waits;
    return wait_rc;
  }
};

#define CHECK(c)                                            \
  do {                                                      \
    if (!(c)) {                                             \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);   \
      return 1;                                             \
    }                                                       \
  } while (0)

static int free_slots(SlotSet& set) {
  std::vector<int> got;
  for (int i; (i = set.take()) >= 0;) got.push_back(i);
  for (int i : got) set.give(i);
  return (int)got.size();
}

int main() {
  SlotSet set;
  CHECK(free_slots(set) == SlotSet::kSlots);
  {  // returned before anything was queued: free at once, nothing to wait for
    SlotLease<Wait> l{Wait{}};
    CHECK(l.take(set) == 0 && free_slots(set) == SlotSet::kSlots - 1);
  }
  CHECK(waits == 0 && free_slots(set) == SlotSet::kSlots);
  {  // the ordinary call: one wait, by the caller
    SlotLease<Wait> l{Wait{}};
    l.take(set);
    l.queued();
    CHECK(l.wait() == 0);
  }
  CHECK(waits == 1 && free_slots(set) == SlotSet::kSlots);
  {  // an early return with work queued waits before the slot is free
    SlotLease<Wait> l{Wait{}};
    l.take(set);
    l.queued();
  }
  CHECK(waits == 2 && free_slots(set) == SlotSet::kSlots);
  wait_rc = 1;
  {  // neither wait succeeds: the queued work may still run, so the slot is not handed on
    SlotLease<Wait> l{Wait{}};
    CHECK(l.take(set) == 0);
    l.queued();
    CHECK(l.wait() == 1);
  }
  CHECK(waits == 4 && free_slots(set) == SlotSet::kSlots - 1);
  wait_rc = 0;
  {
    SlotLease<Wait> l{Wait{}};
    CHECK(l.take(set) == 1);
  }
  // all taken: none, and nothing is given back for it
  std::vector<int> rest;
  for (int i; (i = set.take()) >= 0;) rest.push_back(i);
  {
    SlotLease<Wait> l{Wait{}};
    CHECK(l.take(set) == -1);
    l.queued();
  }
  CHECK(set.take() == -1);
  for (int i : rest) set.give(i);
  // one holder per slot across threads
  std::atomic<int> holder[SlotSet::kSlots] = {}, clashes{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([&] {
      for (int n = 0; n < 20000; ++n) {
        const int i = set.take();
        if (i < 0) continue;
        if (holder[i].fetch_add(1) != 0) ++clashes;
        holder[i].fetch_sub(1);
        set.give(i);
      }
    });
  for (auto& t : ts) t.join();
  CHECK(clashes == 0);
  std::printf("slots ok\n");
  return 0;
}
