"""Sweeps whose wavefronts take turns (1 to 8 wavefronts per SIMD, 24,000 ticks
or more), against the oracle on slices of the grid: outputs of every kind that
parks its state between chunks of ticks, with several steps a sample, orbits
that leave the bound on the way (in the middle and at the ends of chunks) and
orbits that settle.  Everything compared is bit-exact by design."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 257^2 points: 1033 wavefronts, the last group of 64 with 1 point
@pytest.mark.parametrize("sem", [0, 1])
@pytest.mark.parametrize("pre,tmax", [(1, 150.0), (2, 300.02), (3, 450.0)])
@pytest.mark.parametrize("rho,bound", [(24.5, 0.0), (24.5, 17.0), (10.0, 0.0)])
def test_rotating_basins_match_oracle(chaos, oracle, sem, pre, tmax, rho, bound):
    n = 257
    args = (tmax, n, 0.01, [0.0, 0.0, 25.0], [-20.0, 20.0, -20.0, 20.0], [0, 1], 0, bound, 110.0,
            [10.0, rho, 8 / 3], pre)
    print(f"rotating basins sem={sem} pre={pre} rho={rho} bound={bound}", flush=True)
    _, feat, flags = chaos.basins2d(*args, eps=0.5, system="lorenz_rk4", semantics=sem)
    flags, feat = flags.reshape(-1), feat.reshape(feat.shape[0], -1)
    for lo, hi in ((0, 12), (33000, 33024), (n * n - 13, n * n)):
        *want, wfl = oracle.basins_features(oracle.SYS["lorenz_rk4"], sem, *args, point_begin=lo, point_end=hi)
        assert np.array_equal(flags[lo:hi], wfl)
        for k in range(feat.shape[0]):
            assert np.array_equal(feat[k, lo:hi], want[k]), k
    if bound:
        assert 0 < np.count_nonzero(flags == 0) < n * n


def _same_first(c, f, oc, of):
    # the first sample is reported for the points that end at a fixed point
    assert np.array_equal(f[c == -1], of[oc == -1])


# 131,073 points over a span whose steps are powers of two: 2049 wavefronts, and
# every 4096th point is a point of the oracle's 33.  Orbits settle during the
# record (count -1: the first sample, taken 22,000 ticks before, is reported),
# stay chaotic, or leave the bound.
@pytest.mark.parametrize("sem", [0, 1])
@pytest.mark.parametrize("bound", [0.0, 17.0])
def test_rotating_diagram_matches_oracle(chaos, oracle, sem, bound):
    n, coarse = 131073, 33
    args = (0.01, [1.0, 1.0, 1.0], [4.0, 36.0], [1], 0, bound, 15.0, [10.0, 28.0, 8 / 3], 1)
    print(f"rotating diagram sem={sem} bound={bound}", flush=True)
    c, f, pk, iv = chaos.bif1d(225.0, n, *args, system="lorenz_rk4", semantics=sem)
    oc, of, opk, oiv = oracle.bif1d(oracle.SYS["lorenz_rk4"], sem, 225.0, coarse, *args)
    step = (n - 1) // (coarse - 1)
    assert np.array_equal(c[::step], oc)
    _same_first(c[::step], f[::step], oc, of)
    assert (oc == -1).any() and (oc > 0).any() and (bound == 0.0 or (oc == 0).any())
    at = np.concatenate([[0], np.cumsum(np.maximum(c, 0))])
    oat = np.concatenate([[0], np.cumsum(np.maximum(oc, 0))])
    for k in range(coarse):
        p = k * step
        assert np.array_equal(pk[at[p]:at[p + 1]], opk[oat[k]:oat[k + 1]]), k
        assert np.array_equal(iv[at[p]:at[p + 1]], oiv[oat[k]:oat[k + 1]]), k


# the same on a diagram too small to rotate, and with an odd number of samples
@pytest.mark.parametrize("bound", [0.0, 17.0])
@pytest.mark.parametrize("tmax", [225.0, 225.01])
def test_first_samples_match_oracle(chaos, oracle, bound, tmax):
    for sem in (0, 1):
        args = (tmax, 65, 0.01, [1.0, 1.0, 1.0], [4.0, 36.0], [1], 0, bound, 15.0, [10.0, 28.0, 8 / 3], 1)
        print(f"first samples sem={sem} bound={bound}", flush=True)
        c, f, _, _ = chaos.bif1d(*args, system="lorenz_rk4", semantics=sem)
        oc, of, _, _ = oracle.bif1d(oracle.SYS["lorenz_rk4"], sem, *args)
        assert np.array_equal(c, oc) and (oc == -1).any()
        _same_first(c, f, oc, of)
