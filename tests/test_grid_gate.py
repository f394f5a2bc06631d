"""Turns of the grid-mode launches of one device (csrc/sf_grid_gate.h), on the CPU: launches that are
let in together never have more workgroups than the device has CUs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#include "sf_grid_gate.h"

int main()
{
    const int cus = 256;
    {  // many threads, launches of 1 to 256 workgroups
        sf::GridGate gate;
        std::atomic<int> in{0}, worst{0}, together{0};
        std::vector<std::thread> ts;
        for (int t = 0; t < 12; ++t)
            ts.emplace_back([&, t] {
                unsigned r = 1u + t;
                for (int k = 0; k < 300; ++k) {
                    r = r * 1664525u + 1013904223u;
                    const int n = t % 3 ? 1 + (int)(r >> 8) % 60 : 1 + (int)(r >> 8) % 256;
                    gate.enter(n, cus);
                    const int now = in.fetch_add(n) + n;
                    if (now > worst) worst = now;
                    if (now > n) ++together;
                    std::this_thread::sleep_for(std::chrono::microseconds(20));
                    in.fetch_sub(n);
                    gate.leave(n);
                }
            });
        for (auto& t : ts) t.join();
        if (worst > cus || in != 0) return std::printf("%d workgroups at once\n", worst.load()), 1;
        if (together == 0) return std::printf("launches that fit never ran together\n"), 1;
    }
    {  // a launch that has to wait is not passed by a later one that would fit
        sf::GridGate gate;
        std::atomic<int> order{0};
        int large = 0, small = 0;
        gate.enter(200, cus);
        std::thread a([&] { gate.enter(100, cus); large = ++order; gate.leave(100); });
        std::this_thread::sleep_for(std::chrono::milliseconds(100));
        std::thread b([&] { gate.enter(10, cus); small = ++order; gate.leave(10); });
        std::this_thread::sleep_for(std::chrono::milliseconds(100));
        if (order != 0) return std::printf("let in before its turn\n"), 1;
        gate.leave(200);
        a.join();
        b.join();
        if (order != 2) return 1;
    }
    sf::GridGate gate;  // alone, any size
    gate.enter(300, cus);
    gate.leave(300);
    return 0;
}
"""


def test_grid_gate(tmp_path):
    src, exe = tmp_path / "gate.cpp", tmp_path / "gate"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", os.path.join(ROOT, "stokesflow.jl_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
