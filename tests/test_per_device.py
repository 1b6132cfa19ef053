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
