"""Canonical averages at the edges of the kernels' chunks (64 bins, 64
temperatures, four sums or observables side by side) against the oracle, with
ordinary temperatures (E/T as a corrected product) and with T = 0 or energies
beyond 1e100 in the range (E/T as a division), and with infinite and undefined
ln g."""
import numpy as np
import pytest

from oracle import oracle as O
from rewl_simulator_amd.engine import thermo_observables, thermodynamics

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def curve(bins, seed):
    rng = np.random.default_rng(seed)
    x = np.linspace(-1, 1, bins)
    return 200.0 * x, 300.0 * (1 - x * x) + rng.normal(0, 0.1, bins)


def compare(E, lng, N, t0, t1, nT, obs):
    g = thermodynamics(E, lng, N, t0, t1, nT)
    o = O.thermodynamics(E, lng, N, t0, t1, nT)
    # the weights' exp is within 1 ulp on either side, the sums run in the same order
    np.testing.assert_allclose(g[:, :4], o[:, :4], rtol=1e-12, atol=0)
    # C is a difference of U^2 terms: their rounding, amplified by N / T^2
    T = t0 + (t1 - t0) / nT * np.arange(nT)
    with np.errstate(all="ignore"):
        tol = 64 * EPS * N * np.abs(o[:, 2]) / (T * T)
        fine = np.isfinite(o[:, 4])
        assert (np.abs(g[fine, 4] - o[fine, 4]) <= tol[fine] + 1e-12 * np.abs(o[fine, 4])).all()
    np.testing.assert_array_equal(np.isnan(g[:, 4]), np.isnan(o[:, 4]))
    np.testing.assert_allclose(thermo_observables(E, lng, obs, t0, t1, nT), O.thermo_observables(E, lng, obs, t0, t1, nT),
                               rtol=1e-12, atol=0)


@pytest.mark.parametrize("bins", [2, 3, 63, 64, 65, 128, 1000])
@pytest.mark.parametrize("nT,nobs", [(1, 1), (63, 3), (64, 4), (65, 5), (1000, 16)])
def test_chunks(gpu, bins, nT, nobs):
    E, lng = curve(bins, bins)
    obs = np.random.default_rng(nT).random((bins, nobs)) + 0.5
    compare(E, lng, 100, 0.3, 20.0, nT, obs)


@pytest.mark.parametrize("what", ["zero temperature", "negative temperatures", "huge energy", "empty bins", "undefined top",
                                  "undefined inside"])
def test_unusual(gpu, what):
    E, lng = curve(130, 5)
    t0, t1 = 0.5, 8.0
    if what == "zero temperature":
        t0 = 0.0
    elif what == "negative temperatures":
        t0, t1 = -8.0, -0.5
    elif what == "huge energy":
        E[3] = 1e120
    elif what == "empty bins":
        lng[[0, 40, 41, 129]] = -np.inf
    elif what == "undefined top":
        lng[-1] = np.nan
    else:
        lng[70] = np.nan
    obs = np.random.default_rng(1).random((130, 4)) + 0.5
    compare(E, lng, 100, t0, t1, 70, obs)
