"""The exchange kernel against the oracle, bit for bit, over the replica counts
at which its shuffle changes form (one draw more when even, one entry per lane
up to 64) and its wavefronts share out the pairs; the increments' observables."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from rewl_simulator_amd import abi, configs
from rewl_simulator_amd.engine import Engine

from test_gpu_parity import assert_same, window_states_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("obs", [0, 1, 2])
@pytest.mark.parametrize("rng", [abi.RNG_REPLAY, abi.RNG_PHILOX])
@pytest.mark.parametrize("replicas", [1, 2, 3, 16, 17, 63, 64, 65, 128, 255, 256])
def test_exchanges(gpu, replicas, rng, obs):
    N = 36
    s = (configs.at_system(6, -5.0 * N, 0.0, 12.0, 3, replicas) if replicas % 2 else
         configs.ising_system(6, -2.0 * N, 0.0, 4.0, 3, replicas))
    p = configs.params(rng_mode=rng, observables=obs, lnf_initial=0.3, sweeps_per_exchange=1, adjust_mode=1)
    with Engine([s], p) as eng:
        ora = Oracle([s], p)
        eng.adjust_to_range(); ora.adjust_to_range()
        for _ in range(4):
            eng.sweeps(2); ora.sweeps(2)
            eng.exchange(); ora.exchange()
        eng.check(); ora.check()
        eng.exchange(); ora.exchange()
        assert_same(eng, ora, cursors=rng == abi.RNG_REPLAY)
        window_states_equal(eng, ora)
        if not obs:
            return
        corr = eng.correlator_slots(s["model"]) if obs == 2 else []
        for g in range(0, eng.num_walkers, 1 + eng.num_walkers // 40):
            sums = eng.observables(g)
            n = eng.counts(g).astype(np.float64) + eng.visits(g)
            means, counts = ora.observables(g)
            np.testing.assert_array_equal(n, counts, err_msg=f"counts per bin, walker {g}")
            seen = n > 0
            for c in range(sums.shape[1]):
                div = np.ceil(n[seen] / 1000.0) if c in corr else n[seen]
                np.testing.assert_allclose(sums[seen, c] / div, means[seen, c], rtol=1e-9, atol=1e-13,
                                           err_msg=f"walker {g}, column {c}")
