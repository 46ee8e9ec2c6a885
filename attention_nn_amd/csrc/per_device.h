// Set-up that a process does once for each device it launches on (internal).
#pragma once
#include <atomic>

namespace ann {

// A kernel's dynamic-LDS limit is a property of the kernel on one device: set
// on the first, it says nothing about the second.  once() runs `set` (0 for
// success) until it has succeeded on that device; two threads may both run it
// the first time, so it has to be repeatable.  Device ordinals past 63 run it
// every time.
class PerDevice {
 public:
  template <typename F>
  int once(int device, F&& set) {
    const unsigned long long bit = device >= 0 && device < 64 ? 1ull << device : 0;
    if (done_.load(std::memory_order_acquire) & bit) return 0;
    const int e = set();
    if (e == 0) done_.fetch_or(bit, std::memory_order_release);
    return e;
  }

 private:
  std::atomic<unsigned long long> done_{0};
};

}  // namespace ann
