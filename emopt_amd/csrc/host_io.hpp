// Pinned host memory for the results and inputs of a call, and the download of
// large results.  Included by emfdtd.hip.
//
// A copy between device memory and a caller's pageable array goes through the
// runtime's own staging on one thread (8 GB/s for the 9 MB components of a
// 120x80x60 solve).  Here a call borrows a slab of pinned memory: small results
// are written there by the kernel that forms them (no copy operation), and
// large ones are copied in pieces by up to four lanes at once, each a stream
// with two pieces, so that the link, the page faults of the caller's array and
// the host copies overlap.
//
// Slabs belong to the device's pool: at most HOST_SLABS of them, made when
// first needed, lent to one call at a time (a call waits for a free one), and
// given back to the system when the last solver handle of the device goes.
// A call on a device without a handle makes one for itself where that pays (download).
#pragma once

namespace {

constexpr int HOST_LANES = 4;
constexpr int HOST_SLABS = 3;
constexpr size_t HOST_PIECE = size_t(1) << 20;
constexpr size_t HOST_SLAB = HOST_LANES * 2 * HOST_PIECE;

struct HostSlab {
    unsigned char *p = nullptr;
    hipStream_t st[HOST_LANES] = {};
    hipEvent_t ev[HOST_LANES][2] = {};
};

struct HostPool {
    std::mutex m;
    std::condition_variable cv;
    int handles = 0, made = 0;
    std::vector<HostSlab *> idle;
};

constexpr int HOST_DEVICES = 64;
HostPool g_host_pool[HOST_DEVICES];

void slab_free(HostSlab *h)
{
    for (int l = 0; l < HOST_LANES; ++l) {
        for (int q = 0; q < 2; ++q)
            if (h->ev[l][q]) (void)hipEventDestroy(h->ev[l][q]);
        if (h->st[l]) (void)hipStreamDestroy(h->st[l]);
    }
    if (h->p) (void)hipHostFree(h->p);
    delete h;
}

void pool_join(int dev)
{
    HostPool &P = g_host_pool[dev];
    std::lock_guard<std::mutex> lk(P.m);
    ++P.handles;
}

void pool_leave(int dev)
{
    HostPool &P = g_host_pool[dev];
    std::vector<HostSlab *> gone;
    {
        std::lock_guard<std::mutex> lk(P.m);
        if (--P.handles > 0) return;
        gone.swap(P.idle);
        P.made -= (int)gone.size();
    }
    for (HostSlab *h : gone) slab_free(h);
}

// Whether a slab made now outlives the call that asks for it.
bool pool_kept(int dev)
{
    HostPool &P = g_host_pool[dev];
    std::lock_guard<std::mutex> lk(P.m);
    return P.handles > 0;
}

// A slab borrowed from a device's pool for one call (the device is current).
struct HostLoan {
    HostPool *P = nullptr;
    HostSlab *h = nullptr;
    int take(int dev)
    {
        HostPool &pool = g_host_pool[dev];
        {
            std::unique_lock<std::mutex> lk(pool.m);
            pool.cv.wait(lk, [&] { return !pool.idle.empty() || pool.made < HOST_SLABS; });
            P = &pool;
            if (!pool.idle.empty()) {
                h = pool.idle.back();
                pool.idle.pop_back();
                return EMF_OK;
            }
            ++pool.made;
        }
        h = new HostSlab();
        bool ok = hipHostMalloc((void **)&h->p, HOST_SLAB, hipHostMallocDefault) == hipSuccess;
        if (!ok) h->p = nullptr;
        for (int l = 0; l < HOST_LANES && ok; ++l) {
            ok = hipStreamCreateWithFlags(&h->st[l], hipStreamNonBlocking) == hipSuccess;
            for (int q = 0; q < 2 && ok; ++q)
                ok = hipEventCreateWithFlags(&h->ev[l][q], hipEventDisableTiming) == hipSuccess;
        }
        if (!ok) {
            (void)hipGetLastError();
            slab_free(h);
            h = nullptr;
            std::lock_guard<std::mutex> lk(pool.m);
            --pool.made;
            P = nullptr;
            pool.cv.notify_one();
            EMF_FAIL(EMF_ERR_NOMEM, "no pinned host memory");
        }
        return EMF_OK;
    }
    ~HostLoan()
    {
        if (!P) return;
        HostSlab *spare = nullptr;
        {
            std::lock_guard<std::mutex> lk(P->m);
            if (P->handles > 0) P->idle.push_back(h);
            else { spare = h; --P->made; }
        }
        if (spare) slab_free(spare);
        P->cv.notify_one();
    }
};

// f(t) for t = 0 .. n - 1, each in a thread of its own where there is one
template <class F>
void in_threads(int n, F &&f)
{
    std::vector<std::thread> pool;
    int started = 1;
    try {
        for (; started < n; ++started) pool.emplace_back([&f, t = started] { f(t); });
    } catch (const std::exception &) {
        // no more threads, or no memory for one: the rest run here
    }
    f(0);
    for (int t = started; t < n; ++t) f(t);
    for (auto &t : pool) t.join();
}

// threads for `bytes` of host work: one below 2 MB, where starting more costs what they save
int io_threads(size_t bytes)
{
    return (int)std::min<size_t>(HOST_LANES, std::max<size_t>(1, bytes >> 20));
}

// From where on a call on a device without a handle makes a slab of its own, which
// costs 1.05 ms to make and free: 240x120 cells (0.46 MB) take 0.19 ms without and
// 1.25 with one, 240x120x80 (37 MB) 3.8 and 2.6 ms.
constexpr size_t HOST_ALONE = size_t(16) << 20;

// Device memory to a host array.  The work that writes `src` is on stream `st`.
int download(int dev, hipStream_t st, void *dst, const void *src, size_t bytes)
{
    if (bytes < HOST_ALONE && !pool_kept(dev)) {
        HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        return EMF_OK;
    }
    HostLoan loan;
    CHECK(loan.take(dev));
    HostSlab &h = *loan.h;
    if (bytes <= HOST_PIECE) {
        HIPCHK(hipMemcpyAsync(h.p, src, bytes, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        memcpy(dst, h.p, bytes);
        return EMF_OK;
    }
    HIPCHK(hipStreamSynchronize(st));
    const int n = io_threads(bytes);
    std::atomic<int> bad{ 0 };
    in_threads(n, [&](int t) {
        size_t lo = bytes * t / n, hi = bytes * (t + 1) / n;
        lo &= ~size_t(4095);
        if (t + 1 < n) hi &= ~size_t(4095);
        if (hipSetDevice(dev) != hipSuccess) { bad = 1; return; }
        unsigned char *buf[2] = { h.p + 2 * t * HOST_PIECE, h.p + (2 * t + 1) * HOST_PIECE };
        size_t sent = lo, got = lo;
        bool fine = true;
        for (int q = 0; got < hi && fine; ++q) {
            // up to two pieces under way
            for (; fine && sent < hi && sent - got < 2 * HOST_PIECE; sent += std::min(HOST_PIECE, hi - sent)) {
                const int b = (int)(((sent - lo) / HOST_PIECE) & 1);
                fine = hipMemcpyAsync(buf[b], (const char *)src + sent, std::min(HOST_PIECE, hi - sent),
                                      hipMemcpyDeviceToHost, h.st[t]) == hipSuccess &&
                       hipEventRecord(h.ev[t][b], h.st[t]) == hipSuccess;
            }
            const size_t len = std::min(HOST_PIECE, hi - got);
            fine = fine && hipEventSynchronize(h.ev[t][q & 1]) == hipSuccess;
            if (fine) memcpy((char *)dst + got, buf[q & 1], len);
            got += len;
        }
        if (!fine) bad = 1;
        (void)hipStreamSynchronize(h.st[t]);
    });
    if (bad) EMF_FAIL(EMF_ERR_HIP, "download failed: %s", hipGetErrorString(hipGetLastError()));
    return EMF_OK;
}

}  // namespace
