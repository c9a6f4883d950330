"""Admission of kernels whose workgroups wait for each other (csrc/coop.hpp), on the CPU: what is in flight
never exceeds the total, a request for more than the total runs alone, requests are granted in order, and
everyone gets through."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "coop.hpp"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
using namespace lsx;
int main() {
    const int cus = 256, total = coop_cus(cus), dev = 3;
    std::atomic<int> used{0}, peak{0}, bad{0}, done{0};
    std::vector<std::thread> th;
    const int widths[] = {128, 128, 120, 2, 16, 256, 64, 1, 240, 33};
    for (int i = 0; i < 20; ++i)
        th.emplace_back([&, i] {
            const int k = widths[i % 10], eff = k <= 1 ? 0 : (k < total ? k : total);
            for (int r = 0; r < 50; ++r) {
                CoopHold h;
                h.take(dev, cus, k);
                const int u = used.fetch_add(eff) + eff;
                int p = peak.load();
                while (u > p && !peak.compare_exchange_weak(p, u)) {}
                if (u > total) bad++;
                std::this_thread::sleep_for(std::chrono::microseconds(50 * (i % 3)));
                used.fetch_sub(eff);
            }
            done++;
        });
    for (auto& t : th) t.join();
    // in order: a wide request that waits is not overtaken by a later narrow one
    std::atomic<int> order{0}, wide{0}, narrow{0};
    std::thread a, b;
    {
        CoopHold h;
        h.take(dev, cus, 200);
        a = std::thread([&] { CoopHold w; w.take(dev, cus, 100); wide = ++order; });
        std::this_thread::sleep_for(std::chrono::milliseconds(100));
        b = std::thread([&] { CoopHold n; n.take(dev, cus, 8); narrow = ++order; });
        std::this_thread::sleep_for(std::chrono::milliseconds(100));
        if (order != 0) bad++;
    }
    a.join();
    b.join();
    std::printf("%d %d %d %d\n", bad.load(), done.load(), peak.load(), total);
    return bad == 0 && done == 20 && wide > 0 && narrow > 0 ? 0 : 1;
}
"""


def test_admission(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "t.cpp").write_text(SRC)
    exe = tmp_path / "t"
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "linearsolve.jl_amd", "csrc"),
                    str(tmp_path / "t.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
    bad, done, peak, total = (int(v) for v in out.stdout.split())
    assert bad == 0 and done == 20 and 128 < peak <= total == 240
