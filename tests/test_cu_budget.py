"""The budget of compute units that one-launch solves share (csrc/cu_budget.h), compiled with
the host compiler: requests are served in order, so that a large one is not kept out by
small ones that would fit beside what is running, and every request is served."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "shiokaze_amd" / "csrc"

PROGRAM = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#include "cu_budget.h"
int main() {
    shk::CuBudget b;
    std::atomic<int> order{0}, large{0}, small{0}, asked{0};
    b.acquire(200, 256);
    std::thread l([&] { ++asked; b.acquire(256, 256); large = ++order; b.release(256); });
    while (!asked) std::this_thread::yield();
    std::this_thread::sleep_for(std::chrono::milliseconds(100));
    std::thread s([&] { b.acquire(10, 256); small = ++order; b.release(10); });
    std::this_thread::sleep_for(std::chrono::milliseconds(100));
    const bool overtook = small != 0;
    b.release(200);
    l.join();
    s.join();
    // many threads of mixed sizes: never more than the budget, and all are served
    std::atomic<int> used{0}, most{0}, served{0};
    std::vector<std::thread> ts;
    for (int t = 0; t < 12; ++t)
        ts.emplace_back([&, t] {
            for (int k = 0; k < 200; ++k) {
                const int n = 1 + (37 * t + 101 * k) % 256;
                b.acquire(n, 256);
                const int u = used += n;
                for (int m = most; u > m && !most.compare_exchange_weak(m, u);) {}
                used -= n;
                b.release(n);
                ++served;
            }
        });
    for (auto &t : ts) t.join();
    std::printf("%d %d %d %d %d\n", (int)overtook, (int)large, (int)small, (int)most, (int)served);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_requests_are_served_in_order(tmp_path):
    (tmp_path / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", "t.cpp", "-o", "t", "-pthread"], cwd=tmp_path, check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=60, check=True)
    overtook, large, small, most, served = map(int, r.stdout.split())
    assert not overtook and (large, small) == (1, 2)
    assert most <= 256 and served == 12 * 200
