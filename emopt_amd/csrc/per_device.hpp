// Host state kept per device.  Plain C++, no HIP: tested on the CPU.
#pragma once

#include <condition_variable>
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

constexpr int RES_XCDS = 8;

// Admission of resident launches to a device.  All work-groups of the launches
// under way have to run at once, a CU each, and the dispatcher deals those of a
// launch to the XCDs in turn, whatever runs there: a launch of b takes up to
// ceil(b / 8) CUs of any XCD, so it is these that are counted, against the CUs
// of an XCD (100 and 156 work-groups are 256 together, but 13 + 20 on one XCD of
// 32).  A launch alone is always admitted: its planner keeps to the CUs there
// are.  In order of arrival, so that a launch that needs them all is not passed
// by smaller ones for ever.
class ResGate {
    std::mutex m;
    std::condition_variable cv;
    int used = 0, ncu = 0;                       // CUs taken of each XCD; CUs of the device
    unsigned long long next = 0, turn = 0;       // tickets

public:
    static int share(int boxes) { return (boxes + RES_XCDS - 1) / RES_XCDS; }

    // CUs of the device, by ask(&n) the first time it succeeds (returns 0)
    template <class F>
    int cus(int *n, F &&ask)
    {
        std::lock_guard<std::mutex> lk(m);
        int v = ncu;
        const int rc = v ? 0 : ask(&v);
        if (rc == 0) ncu = v;
        *n = ncu;
        return rc;
    }
    void take(int boxes)
    {
        const int c = share(boxes);
        std::unique_lock<std::mutex> lk(m);
        const unsigned long long mine = next++;
        cv.wait(lk, [&] { return turn == mine && (used == 0 || used + c <= ncu / RES_XCDS); });
        used += c;
        ++turn;
        cv.notify_all();
    }
    void give(int boxes)
    {
        { std::lock_guard<std::mutex> lk(m); used -= share(boxes); }
        cv.notify_all();
    }
};

// A launch's admission, given back at the latest with the object.
class ResHold {
    ResGate *g = nullptr;
    int n = 0;

public:
    void take(ResGate &gate, int boxes)
    {
        gate.take(boxes);
        g = &gate;
        n = boxes;
    }
    void give()
    {
        if (g) g->give(n);
        g = nullptr;
    }
    ~ResHold() { give(); }
};

}  // namespace emf
