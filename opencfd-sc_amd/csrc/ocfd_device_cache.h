// ocfd_device_cache.h -- a value per device that every caller would compute
// alike (workgroups resident at once), looked up on first use.  Handles on
// different threads share it.
#pragma once
#include <atomic>

namespace ocfd {

class DeviceCache {
 public:
  static constexpr int DEVICES = 64;
  // `query()`, not 0, the first time; two threads may both ask, for the same value
  template <typename F>
  int get(int dev, F &&query) {
    std::atomic<int> &slot = v_[dev >= 0 && dev < DEVICES ? dev : 0];
    int x = slot.load(std::memory_order_relaxed);
    if (x == 0) {
      x = query();
      slot.store(x, std::memory_order_relaxed);
    }
    return x;
  }

 private:
  std::atomic<int> v_[DEVICES] = {};
};

}  // namespace ocfd
