"""The sixteen-lanes-a-walker sweep (integer energies, Philox) against the
oracle, bit for bit: lattice sizes around its blocks of four sites and its
dword of four blocks, groups whose last wavefront is partly empty, windows of
different widths, couplings and bin sizes at the ends of its byte scales."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from rewl_simulator_amd import abi, configs
from rewl_simulator_amd.engine import Engine

from test_gpu_parity import assert_same, window_states_equal

pytestmark = pytest.mark.gpu


def run_both(systems, sweeps=6, **kw):
    p = configs.params(flatness_mode=abi.FLAT_MIN_OVER_MEAN, flatness=0.3, schedule=abi.SCHED_HALVE,
                       sweeps_per_check=2 * sweeps, sweeps_per_exchange=sweeps, **kw)
    with Engine(systems, p) as eng:
        ora = Oracle(systems, p)
        eng.adjust_to_range(); ora.adjust_to_range()
        for k in range(3):
            eng.sweeps(1 + k); ora.sweeps(1 + k)
            eng.sweeps(sweeps); ora.sweeps(sweeps)
            eng.exchange(); ora.exchange()
            eng.check(); ora.check()
        assert_same(eng, ora, cursors=False)
        window_states_equal(eng, ora)


def ising(L, windows=2, replicas=3, bin=4.0, **kw):
    N = L * L
    return configs.ising_system(L, -2.0 * N, -2.0 * N + bin * np.ceil(2.0 * N / bin), bin, windows, replicas, **kw)


def ashkin_teller(L, windows=2, replicas=3, bin=8.0, **kw):
    N = L * L
    return configs.at_system(L, -5.0 * N, -5.0 * N + bin * np.ceil(5.0 * N / bin), bin, windows, replicas, **kw)


@pytest.mark.parametrize("L", [5, 6, 7, 8, 9, 12, 13, 16, 17, 19, 20, 31, 33, 42, 61, 63, 64])
@pytest.mark.parametrize("model", ["ising", "at"])
def test_sizes(gpu, model, L):
    run_both([(ising if model == "ising" else ashkin_teller)(L, windows=3 if L < 40 else 12)])


@pytest.mark.parametrize("replicas", [1, 2, 5, 7, 64])
@pytest.mark.parametrize("windows", [1, 3])
def test_group_tails(gpu, windows, replicas):
    run_both([ising(10, windows, replicas)])


@pytest.mark.parametrize("walkers", [1030, 2100])
def test_more_walker_wavefronts(gpu, walkers):
    """Two and four walker wavefronts per workgroup."""
    run_both([ising(9, 10, (walkers + 9) // 10)], sweeps=3)


@pytest.mark.parametrize("J,bin", [(1.0, 1.0), (1.0, 2.0), (1.0, 64.0), (1.0, 256.0), (-1.0, 4.0), (3.0, 4.0), (16.0, 4.0),
                                   (40.0, 32.0)])
def test_ising_scales(gpu, J, bin):
    N = 100
    s = ising(10, 2, 3, bin)
    s.update(J=J, e_min=-2.0 * N * abs(J), e_max=-2.0 * N * abs(J) + bin * np.ceil(2.0 * N * abs(J) / bin))
    if (s["e_max"] - s["e_min"]) / bin > 2000:
        s["num_windows"] = 8
    run_both([s])


@pytest.mark.parametrize("J,K", [(1.0, 1.0), (1.0, -0.5), (0.5, 1.0), (2.0, 3.0), (1.0, 0.0), (0.0, 1.0)])
def test_ashkin_teller_couplings(gpu, J, K):
    N = 64
    s = ashkin_teller(8, 2, 3)
    lo = -float(2 * N * (2 * abs(J) + abs(K)))
    s.update(J=J, K=K, e_min=lo, e_max=lo + 8.0 * np.ceil(-lo / 8.0) + 8.0)
    run_both([s], adjust_mode=1)


def test_mixed_context(gpu):
    """Systems of both models and several sizes in one context, one of them
    (E = -1 reachable, a window bound at 0) left to the other kernels."""
    half = ising(9, 2, 3, 1.0, J=0.5, seed=3)
    half.update(e_min=-81.0, e_max=0.0)
    run_both([ising(16, 3, 2), ashkin_teller(11, 2, 5, seed=5), ising(24, 4, 3, 8.0, seed=7), half])
