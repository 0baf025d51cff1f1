"""The one-launch solves' budget of compute units (shyhip_budget.h), compiled
on its own: whatever the order in which solves of 1 .. 8 workgroups to a unit
take and give back their shares, one that needs the whole budget is admitted
afterwards, and concurrent holders never exceed it."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "shyfemcm-ismar_amd", "csrc")

DRIVER = r"""
#include "shyhip_budget.h"
#include <atomic>
#include <cstdio>
#include <random>
#include <thread>
#include <vector>
using namespace shy;
int main() {
    const int units = 256;
    const long cap = unit_budget(units);
    // one workgroup to a unit: 224 of them are the whole budget of 256 units
    if (unit_parts(224, 1) != cap || unit_parts(225, 1) <= cap) return 1;
    for (int occ = 1; occ <= 8; occ++)
        if (unit_parts(3 * occ, occ) != 3 * kUnitParts) return 2;
    UnitBudget b;
    double in_doubles = 0.;                 // the same sequence of shares as real numbers
    std::mt19937 rng(1);
    std::vector<std::pair<int, int>> held;
    long sum = 0;
    for (int i = 0; i < 200000; i++) {
        const int occ = 1 + rng() % 8, nwg = 1 + rng() % 200;
        if (rng() % 2 && sum + unit_parts(nwg, occ) <= cap) {
            b.take(0, unit_parts(nwg, occ), cap);
            in_doubles += (double)nwg / occ;
            sum += unit_parts(nwg, occ);
            held.push_back({nwg, occ});
        } else if (!held.empty()) {
            std::swap(held[rng() % held.size()], held.back());
            const auto h = held.back();
            held.pop_back();
            b.give(0, unit_parts(h.first, h.second));
            in_doubles -= (double)h.first / h.second;
            sum -= unit_parts(h.first, h.second);
        }
    }
    for (const auto &h : held) {
        b.give(0, unit_parts(h.first, h.second));
        in_doubles -= (double)h.first / h.second;
    }
    if (in_doubles == 0.) return 3;         // real numbers do not return to zero
    b.take(0, cap, cap);                    // returns
    b.give(0, cap);
    std::atomic<long> now{0};
    std::atomic<int> bad{0};
    std::vector<std::thread> th;
    for (int t = 0; t < 6; t++)
        th.emplace_back([&, t] {
            std::mt19937 r(t);
            for (int i = 0; i < 2000; i++) {
                const long n = unit_parts(1 + r() % 224, 1 + r() % 8);
                b.take(0, n, cap);
                if ((now += n) > cap) bad++;
                now -= n;
                b.give(0, n);
            }
        });
    for (auto &x : th) x.join();
    b.take(0, cap, cap);
    std::printf("ok %g\n", in_doubles);
    return bad ? 4 : 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_budget_is_whole_again(tmp_path):
    src = tmp_path / "budget.cpp"
    src.write_text(DRIVER)
    exe = str(tmp_path / "budget")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)
