"""The host state that is kept per device (emopt_amd/csrc/per_device.hpp), built
with the host compiler and driven by threads (CPU only)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "emopt_amd", "csrc")
CXX = shutil.which("g++") or shutil.which("c++")

pytestmark = pytest.mark.skipif(CXX is None, reason="no host C++ compiler")


def _run(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text("""
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <thread>
#include <vector>
#include "per_device.hpp"
using namespace emf;
#define EXPECT(c) do { if (!(c)) { std::printf("line %d: %s\\n", __LINE__, #c); return 1; } } while (0)
""" + body)
    exe = str(tmp_path / "t")
    r = subprocess.run([CXX, "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_set_up_runs_before_any_caller_returns_and_on_each_device(tmp_path):
    _run(tmp_path, """
int main()
{
    OncePerDevice once;
    std::atomic<int> calls[2]{}, ready[2]{}, early{ 0 };
    std::vector<std::thread> pool;
    for (int t = 0; t < 8; ++t)
        pool.emplace_back([&, t] {
            const int dev = t & 1;
            once.run(dev, [&] {
                ++calls[dev];
                std::this_thread::sleep_for(std::chrono::milliseconds(50));
                ready[dev] = 1;
                return 0;
            });
            if (!ready[dev]) ++early;
        });
    for (auto &t : pool) t.join();
    EXPECT(early == 0);
    EXPECT(calls[0] == 1 && calls[1] == 1);
    // a failure is reported and tried again
    int tries = 0;
    EXPECT(once.run(63, [&] { ++tries; return 7; }) == 7);
    EXPECT(once.run(63, [&] { ++tries; return 0; }) == 0);
    EXPECT(once.run(63, [&] { ++tries; return 0; }) == 0);
    EXPECT(tries == 2);
    return 0;
}
""")


def test_gate_counts_work_groups_by_xcd_and_admits_in_order(tmp_path):
    _run(tmp_path, """
using ms = std::chrono::milliseconds;
int main()
{
    ResGate g;
    int n = 0;
    EXPECT(g.cus(&n, [](int *v) { *v = 256; return 3; }) == 3 && n == 0);
    EXPECT(g.cus(&n, [](int *v) { *v = 256; return 0; }) == 0 && n == 256);
    EXPECT(g.cus(&n, [](int *v) { *v = 1; return 0; }) == 0 && n == 256);
    // 100 + 156 = 256, but 13 + 20 CUs of the first XCDs
    ResHold a;
    a.take(g, 100);
    std::atomic<int> order{ 0 };
    int b_at = 0, c_at = 0;
    std::thread tb([&] { ResHold h; h.take(g, 156); b_at = ++order; });
    std::this_thread::sleep_for(ms(100));
    // 8 would fit beside the first, but came after
    std::thread tc([&] { ResHold h; h.take(g, 8); c_at = ++order; });
    std::this_thread::sleep_for(ms(100));
    EXPECT(order == 0);
    a.give();
    tb.join(); tc.join();
    EXPECT(b_at == 1 && c_at == 2);
    // 96 + 160 fit side by side
    ResHold d, e;
    d.take(g, 96);
    e.take(g, 160);
    d.give(); e.give();
    // alone, all of them, also where the CUs are no multiple of the XCDs
    ResGate odd;
    odd.cus(&n, [](int *v) { *v = 20; return 0; });
    ResHold f;
    f.take(odd, 20);
    return 0;
}
""")
