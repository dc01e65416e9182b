"""Admission of resident team launches (pp_gate.hpp), compiled for the host: launches that fit run side by side,
never more workgroups than the device holds, and a launch of the whole device gets its turn."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "phipict_amd" / "csrc"
SOURCE = r"""
#include "pp_gate.hpp"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
using namespace pp;
constexpr int CAP = 256;
int main() {
    {   // two launches of 40 and 200 workgroups are inside together: each waits for the other there
        TeamGate g;
        std::atomic<int> inside{0};
        std::atomic<bool> met{false};
        auto one = [&](int need) {
            g.enter(need, CAP);
            if (++inside == 2) met = true;
            const auto end = std::chrono::steady_clock::now() + std::chrono::seconds(10);
            while (!met && std::chrono::steady_clock::now() < end) std::this_thread::yield();
            --inside;
            g.leave(need);
        };
        std::thread a(one, 40), b(one, 200);
        a.join();
        b.join();
        std::printf("%d\n", int(met));
    }
    {   // many threads: the sum stays within the device; a thread that needs all of it comes through
        TeamGate g;
        std::atomic<int> used{0}, worst{0}, whole{0};
        std::vector<std::thread> ts;
        for (int k = 0; k < 8; ++k)
            ts.emplace_back([&, k] {
                for (int i = 0; i < 2000; ++i) {
                    const int need = k == 0 ? CAP : 1 + (k * 37 + i * 11) % 120;
                    g.enter(need, CAP);
                    const int now = used += need;
                    for (int w = worst; now > w && !worst.compare_exchange_weak(w, now);) {}
                    if (k == 0) ++whole;
                    used -= need;
                    g.leave(need);
                }
            });
        for (auto &t : ts) t.join();
        std::printf("%d %d\n", worst.load(), whole.load());
    }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_gate(tmp_path):
    (tmp_path / "gate.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{CSRC}", str(tmp_path / "gate.cpp"), "-o",
                    str(tmp_path / "gate")], check=True)
    out = subprocess.run([str(tmp_path / "gate")], check=True, capture_output=True, text=True, timeout=100).stdout.split()
    assert out[0] == "1", "launches that fit together did not run side by side"
    assert int(out[1]) == 256 and int(out[2]) == 2000
