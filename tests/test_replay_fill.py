"""The replay streams' host side (csrc/replay_fill.hpp), compiled for the host
and run against rings that remember when a copy may still read its words:
every ring holds its stream's words up to its capacity past the cursor, in
order and across the ring's end, and host memory is bounded by the buffer
handed in, however many walkers and however long their streams."""
import os
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r"""
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>
#include "replay_fill.hpp"

struct Copy { int g; uint64_t pos; const uint64_t* w; uint64_t n; };

int main(int argc, char** argv) {
    const int walkers = std::atoi(argv[1]);
    const uint64_t cap = std::strtoull(argv[2], nullptr, 10), room = std::strtoull(argv[3], nullptr, 10);
    std::mt19937_64 moves(7);
    std::vector<std::mt19937_64> engines(walkers);
    std::vector<uint64_t> cursor(walkers, 0), filled(walkers, 0), stage(room), ring(walkers * cap, 0);
    for (int g = 0; g < walkers; ++g) engines[g].seed(g + 1);
    std::vector<Copy> queued;   // started, their words read as late as allowed
    auto finish = [&] {
        for (const Copy& c : queued)
            for (uint64_t k = 0; k < c.n; ++k) ring[c.g * cap + c.pos + k] = c.w[k];
        queued.clear();
        return true;
    };
    std::vector<std::vector<uint64_t>> want(walkers);
    for (int g = 0; g < walkers; ++g) {
        std::mt19937_64 e(g + 1);
        for (uint64_t k = 0; k < 6 * cap; ++k) want[g].push_back(e());
    }
    for (int round = 0; round < 5; ++round) {
        const uint64_t lack = rewl::replay_lack(walkers, cursor.data(), filled.data(), cap);
        uint64_t copied = 0;
        bool bounded = true;
        if (!rewl::replay_fill(
                walkers, cursor.data(), filled.data(), cap, stage.data(), room, [&](int g) { return engines[g](); },
                [&](int g, uint64_t pos, const uint64_t* w, uint64_t n) {
                    bounded = bounded && w >= stage.data() && w + n <= stage.data() + room && pos + n <= cap;
                    copied += n;
                    queued.push_back({g, pos, w, n});
                    return true;
                },
                finish))
            return 2;
        finish();
        if (!bounded || copied != lack) return 3;
        for (int g = 0; g < walkers; ++g) {
            if (filled[g] != cursor[g] + cap) return 4;
            for (uint64_t k = cursor[g]; k < filled[g]; ++k)
                if (ring[g * cap + (k & (cap - 1))] != want[g][k]) return 5;
            cursor[g] += moves() % (cap + 1);
        }
    }
    // a failed copy or wait ends the fill
    if (rewl::replay_fill(
            walkers, cursor.data(), filled.data(), cap, stage.data(), room, [&](int g) { return engines[g](); },
            [](int, uint64_t, const uint64_t*, uint64_t) { return false; }, finish))
        return 6;
    std::puts("ok");
    return 0;
}
"""


@pytest.fixture(scope="module")
def probe():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "probe.cpp"), os.path.join(d, "probe")
        with open(src, "w") as f:
            f.write(PROBE)
        subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-I",
                        os.path.join(ROOT, "rewl_simulator_amd", "csrc"), src, "-o", exe], check=True)
        yield exe


@pytest.mark.parametrize("walkers,cap,room", [(1, 8, 8), (1, 8, 3), (5, 16, 1), (7, 64, 40), (7, 64, 448), (3, 4096, 1000),
                                              (40, 1024, 1024)])
def test_streams_are_filled_through_a_bounded_buffer(probe, walkers, cap, room):
    out = subprocess.run([probe, str(walkers), str(cap), str(room)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.returncode
