"""Per-walker queries gather strided columns into pinned memory: what was set
is what comes back, at window lengths around the gather's block size and for
walkers in the first and last lanes of their groups."""
import numpy as np
import pytest

from rewl_simulator_amd import configs
from rewl_simulator_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [1, 2, 255, 256, 257, 3000])
def test_set_columns_come_back(gpu, bins):
    s = configs.ising_system(64, -8192.0, -8192.0 + 4.0 * bins, 4.0, 1, 70)
    rng = np.random.default_rng(bins)
    with Engine([s], configs.params()) as eng:
        curves = {}
        for g in (0, 1, 63, 64, 69, 0):   # a query after a larger one, and the first walker again
            curves[g] = rng.normal(size=bins)
            eng.set_logdos(g, curves[g])
        spins = np.where(rng.random(4096) < 0.5, 1, -1).astype(np.int8)
        eng.set_spins(69, spins)
        for g, c in curves.items():
            np.testing.assert_array_equal(eng.logdos(g), c)
            assert not eng.counts(g).any() and not eng.visits(g).any()
        np.testing.assert_array_equal(eng.spins(69), spins)
        assert (eng.spins(0) == 1).all() and eng.energy(0) == -8192.0
        eng.set_window_lnf(0, 0.25)
        w = eng.window_info(0)
        assert (w["lnf"], w["iteration"], w["done"], w["one_over_t"]) == (0.25, 1, 0, 0)
