"""GPU online peak detector (chaos_peak_finder) vs the oracle peakFinder:
the hand-traced reference cases plus random quantised signals that exercise
plateaus and the 1e-13 thresholds.  Bit-exact."""
import numpy as np
import pytest

from test_oracle_peaks import HAND_CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("data,peaks,dts", HAND_CASES)
def test_gpu_detector_hand_cases(chaos, data, peaks, dts):
    if len(data) == 0:
        return
    (pk, iv), = chaos.peak_finder(np.array(data, dtype=float), 0.01)
    assert list(pk) == peaks
    assert np.array_equal(iv, np.array(dts, dtype=float) * 0.01)


def test_gpu_detector_random_plateaus(chaos, oracle):
    rng = np.random.default_rng(42)
    rows, n = 512, 400
    steps = rng.choice([0.0, 0.0, 1e-14, -1e-14, 5e-14, -5e-14, 1e-13, 2e-13, -2e-13, 1.0, -1.0, 0.5],
                       size=(rows, n))
    data = np.cumsum(steps, axis=1) + rng.normal(0, 1, (rows, 1))
    print(f"peak_finder rows={rows} n={n}", flush=True)
    got = chaos.peak_finder(data, 0.02)
    for r in range(rows):
        pk, iv = oracle.peak_finder(data[r], 0.02)
        assert np.array_equal(got[r][0], pk), r
        assert np.array_equal(got[r][1], iv), r


# Lorenz up to rho = 30: orbits that spiral into a fixed point until the samples
# differ by rounding only (plateaus, peaks of neighbouring samples), chaotic
# ones, and with a bound of 40 some that leave it on the record.  Every list
# entry is the oracle's, so equality is exact.
@pytest.mark.parametrize("bound", [0.0, 40.0])
@pytest.mark.parametrize("n", [1, 64, 193])
@pytest.mark.parametrize("tmax", [60.0, 60.01])
def test_lists_of_settling_and_leaving_orbits_match_oracle(chaos, oracle, bound, n, tmax):
    for sem in (0, 1):
        args = (tmax, n, 0.01, [1.0, 1.0, 1.0], [3.0, 30.0], [1], 2, bound, 20.0, [10.0, 28.0, 8 / 3], 1)
        print(f"bif1d sem={sem} n={n} tMax={tmax} bound={bound}", flush=True)
        c, f, pk, iv = chaos.bif1d(*args, system="lorenz_rk4", semantics=sem)
        oc, of, opk, oiv = oracle.bif1d(oracle.SYS["lorenz_rk4"], sem, *args)
        assert np.array_equal(c, oc)
        assert np.array_equal(pk, opk) and np.array_equal(iv, oiv)
