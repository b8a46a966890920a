"""Which contexts the sixteen-lanes-a-walker sweep takes (csrc/sweep_choice.hpp,
compiled for the host): at shapes where both kernels were timed, the faster one
(cycles per attempt on 256 CUs with 160 KB of LDS)."""
import os
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r"""
#include <cstdio>
#include <cstdlib>
#include "sweep_choice.hpp"
// planes L observables unrolled walkers | groups lds, one lane's groups lds
int main(int, char** v) {
    auto n = [&](int i) { return std::atoll(v[i]); };
    const long long lds = 163840;
    const int cus = 256;
    bool tree = n(5) <= rewl::tree_walker_limit((int)n(1), (int)n(2), (int)n(3), n(4) != 0);
    if (tree && n(4))
        tree = rewl::tree_pays((int)n(3), rewl::workgroup_rounds(n(6), n(7), lds, cus),
                               rewl::workgroups_per_cu(n(7), lds) == 1, rewl::workgroup_rounds(n(8), n(9), lds, cus));
    std::printf("%d\n", tree ? 1 : 0);
}
"""


@pytest.fixture(scope="module")
def probe():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "probe.cpp"), os.path.join(d, "probe")
        with open(src, "w") as f:
            f.write(PROBE)
        subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-I",
                        os.path.join(ROOT, "rewl_simulator_amd", "csrc"), src, "-o", exe], check=True)
        yield exe


def up(x, k):
    return -(-x // k)


def tree_lds(planes, L, bins, guard, obs):
    """tree_lds of sweep_tree.hpp with rows of 32 bytes a bin."""
    blocks = up(L, 4)
    seg = 1 if L >= 32 else up(32, L)
    at = up(4 * (planes * L * 4 * up(blocks, 4) + 4), 16) * 16 + 4 * (2 * seg * L * 8 + 32) + 4 * 49 * (16 if obs else 8)
    at += 4 * 4 * blocks * 8 if obs == 2 else 0
    n = bins + 2 * guard
    counts = up(max(at, n * 16), 32) * 32
    return 2 * counts + n * 32 + (bins * 32 * (12 if planes == 2 else 3) if obs else 0)


# model, L, bin size, observables, walkers, bins of a window, cycles here, one lane
MEASURED = [
    ("ising", 64, 8, 0, 2048, 118, 110, 159), ("ising", 64, 8, 0, 4096, 217, 124, 160), ("ising", 64, 8, 0, 5120, 179, 152, 164),
    ("ising", 64, 8, 0, 6144, 160, 246, 168), ("ising", 64, 4, 0, 4096, 1171, 220, 319), ("ising", 64, 4, 0, 4096, 1639, 405, 733),
    ("ising", 64, 4, 0, 5120, 1024, 323, 481), ("ising", 32, 4, 0, 4096, 109, 124, 162), ("ising", 32, 4, 0, 4352, 104, 164, 163),
    ("ising", 32, 4, 0, 5120, 90, 166, 162), ("ising", 48, 4, 0, 5120, 202, 148, 168), ("ising", 16, 4, 0, 5120, 24, 172, 176),
    ("at", 64, 8, 0, 4096, 540, 260, 190), ("at", 64, 8, 0, 4352, 512, 263, 190), ("at", 64, 8, 0, 4864, 467, 263, 190),
    ("at", 64, 8, 0, 5120, 447, 263, 396), ("at", 48, 8, 0, 4096, 1152, 236, 401), ("at", 32, 4, 0, 4096, 1024, 251, 402),
    ("ising", 64, 8, 1, 2048, 373, 160, 273), ("ising", 64, 8, 1, 4096, 217, 322, 268), ("ising", 64, 8, 1, 3072, 274, 311, 271),
    ("ising", 64, 8, 1, 2560, 316, 313, 272), ("ising", 64, 8, 1, 4096, 586, 539, 871), ("ising", 64, 8, 1, 4096, 373, 323, 545),
    ("ising", 48, 4, 1, 3072, 308, 310, 273), ("ising", 48, 4, 1, 4096, 244, 320, 583), ("ising", 32, 4, 1, 4096, 293, 374, 584),
    ("ising", 32, 4, 1, 4096, 109, 216, 271), ("at", 32, 16, 1, 4096, 69, 784, 709), ("at", 24, 8, 1, 2560, 112, 768, 649),
    ("at", 24, 8, 1, 4096, 77, 783, 685), ("at", 16, 8, 1, 4096, 93, 806, 1367), ("at", 32, 16, 1, 1024, 184, 298, 764),
    ("at", 48, 16, 1, 4096, 153, 1100, 1260), ("at", 64, 64, 1, 3584, 77, 1066, 627),
    ("at", 64, 32, 1, 4096, 136, 1066, 1230), ("at", 48, 32, 1, 2816, 104, 755, 665),
    ("ising", 64, 8, 2, 4096, 217, 412, 640), ("ising", 64, 8, 2, 4096, 586, 731, 1913), ("at", 32, 16, 2, 4096, 69, 855, 1229),
    ("ising", 5, 4, 0, 6144, 7, 346, 565), ("ising", 5, 4, 0, 7168, 7, 588, 565), ("ising", 7, 4, 0, 10240, 9, 474, 536),
    ("ising", 9, 4, 0, 12288, 12, 530, 521), ("ising", 10, 4, 0, 12288, 15, 481, 517), ("ising", 42, 2, 0, 12288, 1008, 703, 2367),
    ("at", 5, 8, 0, 8192, 7, 804, 681), ("at", 6, 8, 0, 10240, 8, 693, 648), ("at", 9, 8, 0, 10240, 17, 547, 597),
    ("at", 9, 8, 0, 12288, 15, 644, 597), ("at", 14, 8, 0, 12288, 34, 497, 561), ("ising", 20, 8, 1, 4096, 58, 243, 978),
]


@pytest.mark.parametrize("model,L,bin,obs,walkers,bins,here,lane", MEASURED)
def test_the_faster_kernel_is_chosen(probe, model, L, bin, obs, walkers, bins, here, lane):
    planes = 2 if model == "at" else 1
    unrolled = L in (16, 24, 32, 48, 64)
    most = 8 if planes == 1 else 12   # J = 1, K = 1/2
    tl = tree_lds(planes, L, bins, up(4 * most, bin) + 1, obs)
    values = 12 if planes == 2 else 3
    per = (bins + 2 * (up(most, bin) + 1)) * 16 + 16 * L + 16 + (8 * values * bins if obs else 0)
    wide = min(64, (163840 - (16 * L if obs == 2 else 0)) // per)
    out = subprocess.run([probe] + [str(x) for x in (planes, L, obs, int(unrolled), walkers, up(walkers, 4), tl,
                                                     up(walkers, wide), wide * per)],
                         capture_output=True, text=True, check=True)
    assert bool(int(out.stdout)) == (here < lane)
