// pt_once.hpp -- settings made once per device.
#pragma once
#include <atomic>
#include <cstdint>

namespace pt {

// A kernel's attributes belong to the device that is current when they are
// set, so contexts on several devices of one process each need them.  One
// static object per setting; apply(device, set) calls set() the first time for
// each device and returns its result (0: success, others are tried again by
// the next call).  Settings are idempotent: threads that meet here may both
// call set().
class OncePerDevice {
  std::atomic<uint64_t> done_{0};   // devices 0..63; beyond, set() is called every time

 public:
  template <class Set>
  int apply(int device, Set set) {
    const uint64_t bit = device >= 0 && device < 64 ? uint64_t(1) << device : 0;
    if (done_.load(std::memory_order_acquire) & bit) return 0;
    const int rc = set();
    if (rc == 0) done_.fetch_or(bit, std::memory_order_release);
    return rc;
  }
};

}  // namespace pt
