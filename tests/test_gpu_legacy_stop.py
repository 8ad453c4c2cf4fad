"""The legacy windows' early stop in the Lyapunov spectrum and exponent
kernels: trajectories step together while the wavefront is inside the
divergence band and one by one from the first step outside it.  Bounds that
stop some trajectories of a point and not others, a bound that the sum of the
magnitudes passes and no single one does, and windows of one and two steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

IC, VALUES = [1.0, 1.0, 1.0], [10.0, 28.0, 8 / 3]


@pytest.mark.parametrize("max_value", [12.0, 17.5, 60.0])
@pytest.mark.parametrize("nt", [0.01, 0.02, 0.5])
@pytest.mark.parametrize("n", [2, 67])
def test_spectrum_early_stop_matches_oracle(chaos, oracle, max_value, nt, n):
    print(f"legacy LS early stop maxValue={max_value} NT={nt} n={n}", flush=True)
    rg = [20.0, 40.0]
    got = chaos.legacy_ls(3.0, nt, n, 0.01, 1e-6, IC, rg, [1], 1.0, VALUES, dims=1, maxValue=max_value,
                          system="lorenz_rk4", seed=4)
    want = oracle.legacy_ls(oracle.SYS["lorenz_rk4"], 0, 1, 3.0, nt, n, 0.01, 1e-6, IC, rg, [1], max_value, 1.0,
                            VALUES, 4)
    free = chaos.legacy_ls(3.0, nt, n, 0.01, 1e-6, IC, rg, [1], 1.0, VALUES, dims=1, system="lorenz_rk4", seed=4)
    # the windows' log is the platform's (host or device), the orbits are identical
    assert np.allclose(got, want, rtol=1e-10, atol=1e-12, equal_nan=True)
    if max_value == 60.0:
        assert np.array_equal(got, free)


@pytest.mark.parametrize("sweep_ic", [False, True])
@pytest.mark.parametrize("max_value", [12.0, 30.0])
def test_exponent_early_stop_matches_oracle(chaos, oracle, sweep_ic, max_value):
    print(f"legacy LLE early stop maxValue={max_value} sweep_ic={sweep_ic}", flush=True)
    rg, idx = ([-15.0, 15.0], [0]) if sweep_ic else ([20.0, 40.0], [1])
    got = chaos.legacy_lle(3.0, 0.1, 130, 0.01, 1e-6, IC, rg, idx, 1.0, VALUES, dims=1, maxValue=max_value,
                           sweep_ic=sweep_ic, system="lorenz_rk4", seed=4)
    want = oracle.legacy_lle(oracle.SYS["lorenz_rk4"], 0, 1 if sweep_ic else 0, 1, 3.0, 0.1, 130, 0.01, 1e-6, IC, rg,
                             idx, max_value, 1.0, VALUES, 4)
    assert np.allclose(got, want, rtol=1e-10, atol=1e-12, equal_nan=True)


# Runs that stop everywhere (a bound that nothing passes, orbits that overflow)
# end early, after the transient's first step or in the middle of a window.
@pytest.mark.parametrize("max_value,nt", [(-1.0, 0.5), (0.5, 0.5), (0.0, 2.0)])
@pytest.mark.parametrize("n", [3, 130])
def test_all_trajectories_stopped_matches_oracle(chaos, oracle, max_value, nt, n):
    print(f"legacy, all stopped maxValue={max_value} NT={nt} n={n}", flush=True)
    # maxValue 0 stops at NaN / inf only: steps of 0.5 make every orbit overflow
    h, rg = (0.5, [20.0, 40.0]) if max_value == 0.0 else (0.01, [20.0, 40.0])
    got = chaos.legacy_ls(40 * nt, nt, n, h, 1e-6, IC, rg, [1], 20 * h, VALUES, dims=1, maxValue=max_value,
                          system="lorenz_rk4", seed=4)
    want = oracle.legacy_ls(oracle.SYS["lorenz_rk4"], 0, 1, 40 * nt, nt, n, h, 1e-6, IC, rg, [1], max_value, 20 * h,
                            VALUES, 4)
    assert np.allclose(got, want, rtol=1e-10, atol=1e-12, equal_nan=True)
    got = chaos.legacy_lle(40 * nt, nt, n, h, 1e-6, IC, rg, [1], 20 * h, VALUES, dims=1, maxValue=max_value,
                           system="lorenz_rk4", seed=4)
    want = oracle.legacy_lle(oracle.SYS["lorenz_rk4"], 0, 0, 1, 40 * nt, nt, n, h, 1e-6, IC, rg, [1], max_value,
                             20 * h, VALUES, 4)
    assert np.allclose(got, want, rtol=1e-10, atol=1e-12, equal_nan=True)
