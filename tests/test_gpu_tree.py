"""The sixteen-lanes-a-walker sweep (integer energies, Philox) against the
oracle, bit for bit: lattice sizes around its blocks of four sites and its
dword of four blocks, groups whose last wavefront is partly empty, windows of
different widths, couplings and bin sizes at the ends of its byte scales."""
import ctypes

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


@pytest.mark.parametrize("kernel", [{}, dict(producers=1)])
@pytest.mark.parametrize("L", [5, 8, 13, 16, 30, 64])
@pytest.mark.parametrize("obs", [1, 2])
@pytest.mark.parametrize("model", ["ising", "at"])
def test_observables(gpu, model, obs, L, kernel):
    """The observable sums, and with 2 the correlator samples of a bin's
    updates 0, 1000, 2000, ..., against the oracle's running means, over
    several launches, exchanges and a check; chains and counts bit for bit."""
    s = (ising(L, 3 if L < 20 else 12, 3, 8.0 if L > 40 else 4.0) if model == "ising" else
         ashkin_teller(L, 3 if L < 20 else 24, 2))
    p = configs.params(lnf_initial=0.05, observables=obs, sweeps_per_exchange=20, adjust_mode=1, **kernel)
    # attempts for several samples of a bin where the oracle's time allows
    per = max(2, 12000 // (L * L) // (1 if obs == 2 else 4))
    with Engine([s], p) as eng:
        ora = Oracle([s], p)
        eng.adjust_to_range(); ora.adjust_to_range()
        for k in range(4):
            eng.sweeps(per); ora.sweeps(per)
            eng.sweeps(1); ora.sweeps(1)
            eng.exchange(); ora.exchange()
            if k == 1:
                eng.check(); ora.check()
        assert_same(eng, ora, cursors=False)
        corr = eng.correlator_slots(abi.ISING2D if model == "ising" else abi.ASHKIN_TELLER2D) if obs == 2 else []
        for g in range(eng.num_walkers):
            sums = eng.observables(g)
            n = eng.counts(g).astype(np.float64) + eng.visits(g)
            means, counts = ora.observables(g)
            np.testing.assert_array_equal(n, counts, err_msg=f"counts per bin, walker {g}")
            seen = n > 0
            for c in range(sums.shape[1]):
                div = np.ceil(n[seen] / 1000.0) if c in corr else n[seen]
                np.testing.assert_allclose(sums[seen, c] / div, means[seen, c], rtol=1e-9, atol=1e-13,
                                           err_msg=f"walker {g}, column {c}")
            assert np.all(sums[~seen] == 0)


def test_moments_keep_the_generic_kernels_window_limit(gpu):
    """Off the unrolled-row sizes a window with moments is refused above what
    the generic kernel holds, whatever the number of walkers."""
    for kernel in ({}, dict(producers=1)):
        with pytest.raises(abi.REWLError, match="window too wide"):
            Engine([ising(30, 1, 3, 4.0)], configs.params(observables=1, **kernel))


def free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("model,field", [("ising", False), ("at", False), ("ising", True)])
def test_memory_of_a_context(gpu, model, field):
    """Groups of four walkers share rows: a context holds little more than its
    walkers' histograms (8 + 4 + 8 bytes per bin, and the observables), not a
    row of 64 lanes for each group."""
    s = ising(32, 2, 256, 2.0) if model == "ising" else ashkin_teller(32, 4, 256, 16.0)
    obs = 0 if field or model == "ising" else 2
    if field:
        h = configs.gaussian_strain(32, 0.5, 3)
        lo = -2.0 * 1024 - float(np.abs(h).sum())
        s = configs.ising_system(32, lo, lo + 900 * 3.0, 3.0, 2, 256, field=h)
    with Engine([s], configs.params(observables=obs)):   # whatever the first context sets up
        pass
    before = free_memory()
    with Engine([s], configs.params(observables=obs)) as eng:
        held = before - free_memory()
        bins = sum(s["replicas_per_window"] * w["num_bins"] for w in eng.windows)
    per = 20 + (16 * 8 + 4 if obs else 0)
    # rows are as long as their widest window; the same again is left for it
    # and for the granularity of allocations
    assert held <= 2 * per * bins + (16 << 20)


@pytest.mark.parametrize("model,L,obs,copies,replicas", [
    ("ising", 5, 0, 2, (192, 193)), ("at", 6, 0, 2, (192, 193)), ("ising", 9, 0, 3, (213, 214)), ("at", 16, 0, 2, (160, 161)),
    ("ising", 32, 0, 2, (128, 129)), ("ising", 9, 1, 2, (128, 129)), ("at", 16, 2, 2, (128, 129)),
    ("ising", 64, 1, 1, (192, 193)), ("at", 64, 0, 1, (192, 193))])
def test_on_either_side_of_the_choice(gpu, model, L, obs, copies, replicas):
    """Contexts at and just past what the sixteen-lane sweep takes, by walkers
    or (L = 64) by windows so wide that LDS decides: the chain is the same."""
    for R in replicas:
        s = ising(L, 16, R, 8.0 if L == 64 else 4.0) if model == "ising" else ashkin_teller(L, 16, R)
        systems = [dict(s, seed=77 + k) for k in range(copies)]
        p = configs.params(lnf_initial=0.05, observables=obs, adjust_mode=1)
        with Engine(systems, p) as eng:
            ora = Oracle(systems, p)
            eng.adjust_to_range(); ora.adjust_to_range()
            for _ in range(2):
                eng.sweeps(1); ora.sweeps(1)
                eng.exchange(); ora.exchange()
            window_states_equal(eng, ora)
            for g in range(0, eng.num_walkers, 23):
                assert eng.energy(g) == ora.state(g)["E"], g
                np.testing.assert_array_equal(eng.spins(g), ora.spins(g))
                np.testing.assert_array_equal(eng.logdos(g).view(np.uint64), ora.logdos(g).view(np.uint64))
                np.testing.assert_array_equal(eng.counts(g).astype(np.uint64), ora.counts(g))
