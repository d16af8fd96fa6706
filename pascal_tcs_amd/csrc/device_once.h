// device_once.h -- what is set once per device of a process (a kernel's
// attributes belong to the kernel on one device): no HIP here, so that the
// rule can be tested on any host.
#pragma once

#include <atomic>
#include <cstdint>

namespace tcs {

// The devices, by number, for which something has been done.
struct DeviceSet {
    std::atomic<uint64_t> bits{0};
};

// set() (0: done) unless it has been done for device dev.  Threads that come
// at the same time may each do it; none returns 0 before it is done.
// Devices past the 64th are not remembered: done at every call.
template <class Set>
int once_per_device(DeviceSet &done, int dev, Set set) {
    const uint64_t bit = dev >= 0 && dev < 64 ? (uint64_t)1 << dev : 0;
    if (done.bits.load(std::memory_order_acquire) & bit) return 0;
    const int rc = set();
    if (rc == 0) done.bits.fetch_or(bit, std::memory_order_release);
    return rc;
}

}  // namespace tcs
