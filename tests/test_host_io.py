"""The pool of pinned result memory (emopt_amd/csrc/host_io.hpp), built with the
host compiler against a stand-in for the HIP calls that it makes (CPU only)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "emopt_amd", "csrc")
CXX = shutil.which("g++") or shutil.which("c++")

pytestmark = pytest.mark.skipif(CXX is None, reason="no host C++ compiler")

STAND_IN = r"""
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <exception>
#include <thread>
#include <vector>
typedef int hipError_t;
typedef int *hipStream_t;
typedef int *hipEvent_t;
enum { hipSuccess = 0, hipHostMallocDefault = 0, hipStreamNonBlocking = 1, hipEventDisableTiming = 2,
       hipMemcpyDeviceToHost = 2 };
static std::atomic<int> slabs{ 0 }, streams{ 0 }, events{ 0 }, made{ 0 };
static int hipHostMalloc(void **p, size_t n, int) { *p = malloc(n); ++slabs; ++made; return 0; }
static int hipHostFree(void *p) { free(p); --slabs; return 0; }
static int hipStreamCreateWithFlags(hipStream_t *s, int) { *s = new int; ++streams; return 0; }
static int hipStreamDestroy(hipStream_t s) { delete s; --streams; return 0; }
static int hipEventCreateWithFlags(hipEvent_t *e, int) { *e = new int; ++events; return 0; }
static int hipEventDestroy(hipEvent_t e) { delete e; --events; return 0; }
static int hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
static int hipEventSynchronize(hipEvent_t) { return 0; }
static int hipStreamSynchronize(hipStream_t) { return 0; }
static int hipSetDevice(int) { return 0; }
static int hipGetLastError() { return 0; }
static const char *hipGetErrorString(int) { return ""; }
static int hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) { memcpy(d, s, n); return 0; }
enum { EMF_OK = 0, EMF_ERR_HIP = -2, EMF_ERR_NOMEM = -3 };
#define EMF_FAIL(rc, ...) do { std::printf(__VA_ARGS__); return rc; } while (0)
#define CHECK(x) do { const int rc_ = (x); if (rc_ != EMF_OK) return rc_; } while (0)
#define HIPCHK(x) do { if ((x) != hipSuccess) return EMF_ERR_HIP; } while (0)
#include "host_io.hpp"
#define EXPECT(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
"""


def _run(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text(STAND_IN + body)
    exe = str(tmp_path / "t")
    r = subprocess.run([CXX, "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_downloads_and_the_life_of_slabs(tmp_path):
    """Whole copies at sizes around a piece, a lane's share and odd ends; a slab is
    made for devices with a handle, and given back with the last one; without, for
    the call alone and only where it is large."""
    _run(tmp_path, """
int main()
{
    int st = 0;
    const size_t sizes[] = { 16, HOST_PIECE, HOST_PIECE + 16, 2 * HOST_PIECE - 16, 3 * HOST_PIECE + 4112,
                             HOST_SLAB, 9 * HOST_PIECE + 48, HOST_ALONE - 16, HOST_ALONE };
    for (int handle = 0; handle < 2; ++handle) {
        if (handle) { pool_join(3); pool_join(3); }
        for (size_t n : sizes) {
            std::vector<unsigned char> src(n), dst(n + 64, 7);
            for (size_t q = 0; q < n; ++q) src[q] = (unsigned char)(q * 31 + (q >> 12));
            EXPECT(download(3, &st, dst.data(), src.data(), n) == EMF_OK);
            EXPECT(memcmp(dst.data(), src.data(), n) == 0);
            for (int q = 0; q < 64; ++q) EXPECT(dst[n + q] == 7);
            EXPECT(made == (handle ? 2 : n >= HOST_ALONE) && slabs == handle);
        }
    }
    pool_leave(3);
    EXPECT(slabs == 1);
    pool_leave(3);
    EXPECT(slabs == 0 && streams == 0 && events == 0);
    return 0;
}
""")


def test_a_slab_still_lent_goes_with_its_loan(tmp_path):
    _run(tmp_path, """
int main()
{
    pool_join(0);
    {
        HostLoan a, b, c;
        EXPECT(a.take(0) == EMF_OK && b.take(0) == EMF_OK && c.take(0) == EMF_OK);
        std::atomic<bool> got{ false };
        std::thread t([&] { HostLoan d; d.take(0); got = true; });
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        const bool early = got;
        { HostLoan gone; std::swap(gone.P, a.P); std::swap(gone.h, a.h); }
        t.join();
        EXPECT(!early && slabs == HOST_SLABS);
        pool_leave(0);
    }
    EXPECT(slabs == 0 && streams == 0 && events == 0);
    return 0;
}
""")


def test_work_is_done_where_threads_are_not_to_be_had(tmp_path):
    """Out of memory at each allocation that starting the threads makes."""
    _run(tmp_path, """
#include <new>
static std::atomic<int> left{ -1 };
void *operator new(size_t n)
{
    if (left >= 0 && left-- == 0) throw std::bad_alloc();
    void *p = malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
int main()
{
    for (int at = 0; at < 12; ++at) {
        std::atomic<int> runs[4]{};
        left = at;
        in_threads(4, [&](int t) { ++runs[t]; });
        left = -1;
        for (auto &r : runs) EXPECT(r == 1);
    }
    return 0;
}
""")
