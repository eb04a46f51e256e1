// device_cache.h — launch-size figures looked up once per device and kept for the process (CU
// counts, resident grids). Launchers read them from any host thread, without a lock.
#pragma once
#include <atomic>

namespace vib3 {

// One positive int per device, 0 until it is known. Threads that meet an unknown entry at the same
// time each compute the same value and store it; relaxed order suffices, the value stands alone.
class DeviceCache {
 public:
  template <class Compute>
  int get(int dev, Compute compute) {
    std::atomic<int>& e = entry_[dev & 63];
    int v = e.load(std::memory_order_relaxed);
    if (v == 0) {
      v = compute();
      e.store(v, std::memory_order_relaxed);
    }
    return v;
  }

 private:
  std::atomic<int> entry_[64] = {};
};

}  // namespace vib3
