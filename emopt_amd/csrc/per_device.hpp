// Host state kept per device.  Plain C++, no HIP: tested on the CPU.
#pragma once

#include <mutex>

namespace emf {

constexpr int PER_DEVICE_MAX = 64;

// Runs a set-up call once per device: a caller returns when the call has
// succeeded for its device, also where another thread is making it.  What
// failed is tried again by the next caller.  One for each kernel whose
// attributes have to be set before its first launch on a device.
class OncePerDevice {
    std::mutex m;
    unsigned long long done = 0;

public:
    // f() returns 0 when it has succeeded
    template <class F>
    int run(int dev, F &&f)
    {
        const unsigned long long bit = 1ULL << (dev & (PER_DEVICE_MAX - 1));
        std::lock_guard<std::mutex> lk(m);
        if (done & bit) return 0;
        const int rc = f();
        if (rc == 0) done |= bit;
        return rc;
    }
};

}  // namespace emf
