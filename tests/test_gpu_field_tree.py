"""The sixteen-lanes-a-walker sweep for FP64 energies (Philox) against the
oracle, and the kernel with one lane a walker against the same, bit for bit:
lattice sizes around its blocks of four sites, groups whose wavefront is partly
empty, energies on the edges of bins, windows that touch zero, couplings off
the integers without a field."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from rewl_simulator_amd import abi, configs
from rewl_simulator_amd.engine import Engine

from test_gpu_parity import assert_same, window_states_equal

pytestmark = pytest.mark.gpu

ONE_LANE = dict(producers=1)   # a launch shape of its own keeps one lane a walker


def run_both(systems, sweeps=4, **kw):
    p = configs.params(flatness_mode=abi.FLAT_MIN_OVER_MEAN_VISITED, flatness=0.3, schedule=abi.SCHED_HALVE,
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


def field_system(model, L, windows=2, replicas=3, bins=120, field=None, seed=1, **kw):
    N = L * L
    h = configs.gaussian_strain(L, 0.5, 100 + L) if field is None else field
    lo = -(2.0 if model == "ising" else 5.0) * N - float(np.abs(h).sum())
    bs = -lo / (bins - 1)
    make = configs.ising_system if model == "ising" else configs.at_system
    return make(L, lo, lo + bs * bins, bs, windows, replicas, field=h, seed=seed, **kw)


@pytest.mark.parametrize("L", [5, 6, 7, 8, 9, 12, 13, 16, 17, 30, 31, 32, 33, 48, 63, 64])
@pytest.mark.parametrize("model", ["ising", "at"])
def test_sizes(gpu, model, L):
    run_both([field_system(model, L)],
             adjust_mode=1 if model == "at" else 0)


@pytest.mark.parametrize("L", [16, 24, 32, 48])
@pytest.mark.parametrize("model", ["ising", "at"])
def test_one_lane_unrolled_rows(gpu, model, L):
    run_both([field_system(model, L)], adjust_mode=1 if model == "at" else 0, **ONE_LANE)


@pytest.mark.parametrize("kernel", [{}, ONE_LANE])
@pytest.mark.parametrize("replicas", [1, 2, 5, 64])
@pytest.mark.parametrize("windows", [1, 3])
def test_group_tails(gpu, windows, replicas, kernel):
    run_both([field_system("ising", 10, windows, replicas)], **kernel)


@pytest.mark.parametrize("kernel", [{}, ONE_LANE])
@pytest.mark.parametrize("model", ["ising", "at"])
@pytest.mark.parametrize("L", [9, 16])
def test_energies_on_bin_edges(gpu, model, L, kernel):
    """A field of multiples of 1/2 and bins of 3 or 0.5: quotients at and next
    to integers, so that the division decides."""
    rng = np.random.default_rng(L)
    h = 0.5 * rng.integers(-2, 3, L * L).astype(np.float64)
    for bs in (3.0, 0.5):
        s = field_system(model, L, windows=4 if bs == 3.0 else 12, replicas=2, field=h)
        lo = np.floor(s["e_min"])
        s.update(e_min=lo, e_max=lo + bs * np.ceil(-lo / bs), bin_size=bs)
        run_both([s], adjust_mode=1, **kernel)


@pytest.mark.parametrize("kernel", [{}, ONE_LANE])
def test_couplings_off_the_integers(gpu, kernel):
    N = 100
    a = configs.ising_system(10, -140.0, 0.7, 0.7, 2, 3, J=0.7)
    a.update(e_max=-140.0 + 0.7 * 200)
    b = configs.at_system(8, -64 * 4.6, 0.0, 4.6, 2, 3, J=1.0, K=0.3)
    c = configs.ising_system(11, -2.0 * 121 - 30.25, 0.0, 1.0, 3, 2, seed=5)
    c.update(h=0.25, e_max=-2.0 * 121 - 30.25 + 272.0)
    run_both([a, b, c], adjust_mode=1, **kernel)


def test_mixed_context(gpu):
    """Field systems of both models and several sizes beside an integer one,
    swept for more sweeps than one launch's buffers alternate over."""
    N = 81.0
    clean = configs.ising_system(9, -2 * N, -2 * N + 4.0 * np.ceil(N / 2), 4.0, 2, 3, seed=3)
    run_both([field_system("ising", 13, 2, 2, seed=7), clean, field_system("at", 16, 3, 2, seed=9),
              field_system("at", 7, 2, 5, seed=11)], sweeps=7, adjust_mode=1)


@pytest.mark.parametrize("model", ["ising", "at"])
@pytest.mark.parametrize("more", [0, 1])
def test_on_either_side_of_the_choice(gpu, model, more):
    """4096 walkers of one size, the most that the sixteen-lane sweep takes, and
    a few more: the chain is the same."""
    s = [field_system(model, 9, 4, r, seed=k + 1) for k, r in enumerate([256] * 4 + [1] * more)]
    p = configs.params(lnf_initial=0.05, adjust_mode=1)
    with Engine(s, p) as eng:
        ora = Oracle(s, p)
        eng.adjust_to_range(); ora.adjust_to_range()
        for _ in range(2):
            eng.sweeps(2); ora.sweeps(2)
            eng.exchange(); ora.exchange()
        window_states_equal(eng, ora)
        for g in range(0, eng.num_walkers, 23):
            assert eng.energy(g) == ora.state(g)["E"], g
            np.testing.assert_array_equal(eng.spins(g), ora.spins(g))
            np.testing.assert_array_equal(eng.logdos(g).view(np.uint64), ora.logdos(g).view(np.uint64))
            np.testing.assert_array_equal(eng.counts(g).astype(np.uint64), ora.counts(g))


@pytest.mark.parametrize("kernel", [{}, ONE_LANE])
@pytest.mark.parametrize("model", ["ising", "at"])
@pytest.mark.parametrize("L", [24, 32, 48])
def test_energies_on_bin_edges_of_unrolled_rows(gpu, model, L, kernel):
    """The same on the sides whose rows the kernel with one lane a walker
    unrolls: a field of multiples of 1/2 and bins of 3."""
    h = np.round(2.0 * configs.gaussian_strain(L, 1.0, 200 + L)) / 2.0
    N, span = L * L, float(np.ceil(np.abs(h).sum())) + 8.0
    s = (configs.ising_system(L, -2.0 * N - span, 2.0 * N + span, 3.0, 6, 2, field=h) if model == "ising" else
         configs.at_system(L, -5.0 * N - span, 3.0 * N + span, 3.0, 6, 2, field=h))
    run_both([s], adjust_mode=1 if model == "at" else 0, **kernel)
