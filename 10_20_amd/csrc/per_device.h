// What a process sets once on every device that it uses.
#pragma once
#include <stdint.h>

#include <atomic>

namespace v1 {

// run(device, work) calls `work` (status 0: done) unless it has succeeded for
// that device before; a failure is returned and tried again by the next call.
// Several threads may be the first at a time, so `work` sets the same thing
// whoever does it.  Devices from 64 on are not remembered.
class OncePerDevice {
    std::atomic<uint64_t> done_{0};

  public:
    template <class Work>
    int run(int device, Work work) {
        const uint64_t bit = device >= 0 && device < 64 ? 1ull << device : 0;
        if (done_.load(std::memory_order_acquire) & bit) return 0;
        const int rc = work();
        if (rc == 0) done_.fetch_or(bit, std::memory_order_release);
        return rc;
    }
};

}  // namespace v1
