"""The launch-shape autotuner's choices, with the timing replaced by a table."""
import json

import pytest

from rewl_simulator_amd import abi, autotune, configs

AUTO = dict(walkers_per_group=0, producers=0, sweep_kernel=0)


def workload(kind, L):
    if kind == "field":
        return [configs.ising_system(L, -3.0 * L * L, 0.0, 4.0, 2, 2, field=configs.gaussian_strain(L, 0.5, 1))], {}
    return [configs.ising_system(L, -2.0 * L * L, 0.0, 4.0, 2, 2)], dict(rng_mode=abi.RNG_REPLAY) if kind == "replay" else {}


@pytest.fixture
def rates(monkeypatch):
    table = {}
    monkeypatch.setattr(autotune, "_CACHE", {})
    monkeypatch.setattr(autotune, "measure",
                        lambda systems, params, shape, sweeps: table.get(json.dumps(shape, sort_keys=True), 1.0))
    return table


@pytest.mark.parametrize("kind", ["integer", "field", "replay"])
@pytest.mark.parametrize("L", [8, 16, 42, 64])
def test_the_automatic_shape_is_a_candidate(rates, kind, L):
    """Where it is the fastest it is chosen: an autotuned context is never
    slower than one left alone."""
    systems, p = workload(kind, L)
    params = configs.params(**p)
    shapes = autotune.candidates(systems, params)
    assert shapes[0] == AUTO
    assert len({json.dumps(s, sort_keys=True) for s in shapes}) == len(shapes) > 1
    rates[json.dumps(AUTO, sort_keys=True)] = 2.0
    best, seen = autotune.autotune(systems, params)
    assert best == AUTO and len(seen) == len(shapes)


def test_one_lane_per_walker_remains_a_candidate(rates):
    systems, p = workload("integer", 64)
    one_lane = dict(AUTO, sweep_kernel=3)
    rates[json.dumps(one_lane, sort_keys=True)] = 2.0
    assert autotune.autotune(systems, configs.params(**p))[0] == one_lane
    systems, p = workload("field", 30)
    one_lane = dict(AUTO, producers=1)
    rates[json.dumps(one_lane, sort_keys=True)] = 3.0
    assert autotune.autotune(systems, configs.params(**p))[0] == one_lane


def test_choices_are_kept_per_workload(rates, tmp_path):
    """Observables run other kernels than a run without, and a cache file of
    another version of the candidates is not used."""
    systems, p = workload("integer", 42)
    plain, moments = configs.params(**p), configs.params(observables=1, **p)
    assert len({autotune.signature(systems, q) for q in (plain, moments, configs.params(observables=2, **p))}) == 3
    cache = tmp_path / "shapes.json"
    slow = dict(AUTO, sweep_kernel=1)
    version = autotune.VERSION
    autotune.VERSION = version - 1
    try:
        cache.write_text(json.dumps({autotune.signature(systems, plain): slow}))
    finally:
        autotune.VERSION = version
    rates[json.dumps(AUTO, sort_keys=True)] = 2.0
    best, seen = autotune.autotune(systems, plain, cache_path=str(cache))
    assert best == AUTO and seen
    autotune._CACHE.clear()
    best, seen = autotune.autotune(systems, plain, cache_path=str(cache))   # now from the file
    assert best == AUTO and not seen
