// A setting that has to be made once on every device, such as the dynamic LDS
// limit of a kernel: an attribute belongs to the device that was current when
// it was set.  (No HIP in here: the header is also compiled on the host alone.)
#pragma once
#include <atomic>
#include <cstdint>

namespace d2q9 {

class PerDevice {
 public:
  // Calls set() -- 0 when it succeeds -- unless it has succeeded for `device`
  // before, and returns its code.  A failure is not remembered.  Threads that
  // meet here at first may call set() twice.  Devices from 64 on are always set.
  template <typename F>
  int once(int device, F set) {
    const uint64_t bit = device >= 0 && device < 64 ? uint64_t{1} << device : 0;
    if (done_.load(std::memory_order_acquire) & bit) return 0;
    const int rc = set();
    if (rc == 0) done_.fetch_or(bit, std::memory_order_release);
    return rc;
  }

 private:
  std::atomic<uint64_t> done_{0};
};

}  // namespace d2q9
