"""The step maps' transcendentals on the GPU at the arguments where their
range reduction and quadrant selection can go wrong: single steps of the maps
that call sin / cos (and exp / atan) from states at and around the multiples of
pi/2, across many binades, beyond 2^51 pi/2 (where the multiple of pi/2 no
longer has unit spacing), at zeros, subnormals and the largest finite values,
infinities and NaN -- bit-equal to the oracle (NaN where it is NaN)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def edge_values():
    rng = np.random.default_rng(17)
    k = np.concatenate([np.arange(-40, 41), 2 ** np.arange(6, 62, 3), -(2 ** np.arange(6, 62, 3)) + 1]).astype(float)
    base = k * (np.pi / 2)
    near = np.concatenate([base, np.nextafter(base, np.inf), np.nextafter(base, -np.inf), base + np.pi / 4])
    wide = rng.uniform(1, 2, 2000) * 2.0 ** rng.integers(-1060, 1023, 2000) * rng.choice([-1.0, 1.0], 2000)
    mid = rng.uniform(-400, 400, 2000)
    special = np.array([0.0, -0.0, 5e-324, -5e-324, 2.2e-308, np.inf, -np.inf, np.nan, 1.7e308, -1.7e308,
                        2.0 ** 51, 2.0 ** 52 + 1, 2.0 ** 53 - 1, 2.0 ** 53, 2.0 ** 54 + 4])
    return np.concatenate([near, wide, mid, special])


@pytest.mark.parametrize("system,params,h", [
    ("chameleon", (0.5, 3.0, 0.0, 2.0, 1.0, 18.0, 1.0), 0.01),
    ("chameleon", (0.0, 0.0, 0.5, 1.0, 1.0, 1.0, 0.0), 1.0),
    ("basins", (0.5, 0.1, 1.4, 15.552, 2.0), 0.01),
    ("basins", (1.0, 0.0, 1.4, 15.552, 2.0), 1.0),
    ("basins_2", (0.5, 0.1), 0.01),
    ("damir", (1e-5, 1e5), 1e-10),
])
def test_one_step_bit_exact_at_edge_arguments(chaos, oracle, system, params, h):
    sid = oracle.SYS[system]
    nx, _ = oracle.dims(sid)
    v = edge_values()
    rng = np.random.default_rng(3)
    # the edge value in every component in turn, ordinary values in the others
    X = rng.uniform(-0.5, 0.5, (nx, v.size, nx))
    for j in range(nx):
        X[j, :, j] = v
    X = X.reshape(-1, nx)
    P = np.tile(np.asarray(params, dtype=float), (len(X), 1))
    print(f"one step of {system} {params} h={h} from {len(X)} edge states", flush=True)
    got = chaos.integrate(system, P, X, 1, h)
    want = oracle.integrate(sid, P, X, 1, h)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    bad = (got.view(np.uint64) != want.view(np.uint64)) & ~nan
    assert not bad.any(), (X[bad.any(1)][:3], got[bad.any(1)][:3], want[bad.any(1)][:3])
