"""The arrival word of the in-launch maximum (csrc/grid_word.hpp) on host
threads, one thread per workgroup: ordered launches all see every slot, and
launches that overlap on one word (a misuse) leave it as good as new."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>
#include "grid_word.hpp"

struct State {
    std::atomic<unsigned long long> word{0};
    std::atomic<unsigned> slots[64] = {};
    std::atomic<int> gave_up{0};
};

struct HostWord {
    State* s;
    unsigned long long add(unsigned long long x) const { return s->word.fetch_add(x); }
    void and_(unsigned long long x) const { ++s->gave_up; s->word.fetch_and(x); }
    unsigned long long load() const { return s->word.load(); }
    void pause() const { std::this_thread::yield(); }
};

static unsigned workgroup(State& s, unsigned wg, unsigned nwg, unsigned value, unsigned polls) {
    s.slots[wg].exchange(value);
    ft::grid_arrive(HostWord{&s}, nwg, polls);
    unsigned mx = 0;
    for (unsigned i = 0; i < nwg; ++i) mx = std::max(mx, s.slots[i].load());
    return mx;
}

// launches of the given sizes at once; true when every workgroup of every
// launch saw its launch's largest value
static bool launch(State& s, const std::vector<unsigned>& sizes, unsigned base, unsigned polls) {
    std::vector<std::thread> threads;
    std::atomic<int> wrong{0}, gate{0};
    for (unsigned nwg : sizes)
        for (unsigned wg = 0; wg < nwg; ++wg)
            threads.emplace_back([&, nwg, wg] {
                while (!gate.load()) std::this_thread::yield();
                unsigned top = 0;
                for (unsigned i = 0; i < nwg; ++i) top = std::max(top, base + i * 7 % nwg);
                if (workgroup(s, wg, nwg, base + wg * 7 % nwg, polls) != top) ++wrong;
            });
    gate = 1;
    for (auto& t : threads) t.join();
    return wrong == 0;
}

int main() {
    const unsigned kForever = 1u << 30;
    State s;
    unsigned base = 1000;
    // values fall from launch to launch, so a stale slot would win the maximum
    for (int i = 0; i < 60; ++i, base -= 5)
        for (unsigned nwg : {1u, 2u, 7u, 12u})
            if (!launch(s, {nwg}, base, kForever) || (unsigned)s.word.load() != 0 || s.gave_up)
                return printf("ordered launches: %u workgroups\n", nwg), 1;
    for (int i = 0; i < 60; ++i, base -= 5) {
        launch(s, {5, 9}, base + 2000, 300);  // overlapping: any values, few polls
        if ((unsigned)s.word.load() != 0)
            return printf("%u arrivals left behind\n", (unsigned)s.word.load()), 1;
        s.gave_up = 0;
        for (unsigned nwg : {9u, 5u, 12u})
            if (!launch(s, {nwg}, base, kForever) || s.gave_up)
                return printf("after an overlap: %u workgroups\n", nwg), 1;
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid_word")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(ROOT, "fusedtok_amd", "csrc"), str(d / "main.cpp"), "-o",
                    str(d / "main")], check=True)
    return str(d / "main")


def test_ordered_launches_and_launches_after_an_overlap(program):
    p = subprocess.run([program], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout
