"""Grids between one and eight wavefronts per SIMD: the wavefronts take turns
on the SIMDs, with the lane state parked between chunks of ticks, and small
exponent maps run a point's two trajectories on two lanes.  Results do not
depend on either: compared with the oracle on sampled rows, with the same map
computed in ranges too small to rotate, and with the job server's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROS = dict(values=[0.2, 0.2, 5.7], ic=[0.1, 0.1, 0.1], ranges=[0.05, 0.35, 2.0, 10.0], idx=[0, 2])
CHAM = dict(values=[0.5, 3, 0, 2, 1, 18, 1], ic=[3.0, 3.0, 0.0], ranges=[0.0, 5.0, 0.0, 20.0], idx=[3, 5])
LOR = dict(values=[10.0, 28.0, 8 / 3], ic=[1.0, 1.0, 1.0], ranges=[20.0, 200.0, 0.5, 4.0], idx=[1, 2])


def _lle_rows(chaos, oracle, system, s, n, CT, TT, sem, rows, eps=1e-7):
    print(f"LLE {system} n={n} CT={CT} TT={TT} sem={sem}", flush=True)
    got = chaos.lle2d(CT, 0.5, n, 0.01, eps, s["ic"], s["ranges"], s["idx"], TT, s["values"], system=system,
                      semantics=sem, seed=77)
    for r in rows:
        want = oracle.lle2d(oracle.SYS[system], sem, CT, 0.5, n, 0.01, eps, s["ic"], s["ranges"], s["idx"], TT,
                            s["values"], 77, r, r + 1)
        # the windows' log is the platform's (host or device), the orbits are identical
        err = np.abs(got[r] - np.asarray(want).reshape(-1)[-n:])
        assert err.max() <= 1e-12, (r, err.max())


# 1057 wavefronts rotate one to a SIMD; the last group of 64 is not full
@pytest.mark.parametrize("sem", [0, 1])
def test_rotating_exponent_map_matches_oracle(chaos, oracle, sem):
    _lle_rows(chaos, oracle, "rossler_rk4", ROS, 260, 210.0, 40.0, sem, [0, 131, 259])


# 2 * 200^2 trajectories on 1250 wavefronts: the windows rotate
def test_rotating_lane_pairs_match_oracle(chaos, oracle):
    _lle_rows(chaos, oracle, "chameleon", CHAM, 200, 250.0, 5.0, 0, [0, 100, 199])


@pytest.mark.parametrize("n", [1, 2, 5, 6, 17])
@pytest.mark.parametrize("CT,TT", [(2.0, 0.0), (2.49, 3.0), (7.0, 1.37)])
def test_lane_pairs_match_oracle_at_small_sizes(chaos, oracle, n, CT, TT):
    for system, s in (("rossler_rk4", ROS), ("basins_2", dict(values=[0.5, 0.1], ic=[0.3, -0.2],
                                                              ranges=[0.4, 0.6, 0.05, 0.2], idx=[0, 1]))):
        for sem in (0, 1):
            _lle_rows(chaos, oracle, system, s, n, CT, TT, sem, [0, n - 1])


@pytest.mark.parametrize("system,s,sem", [("lorenz_rk4", LOR, 1), ("chameleon", CHAM, 0), ("lorenz_rk4", LOR, 0)])
def test_rotating_peak_map_equals_ranges(chaos, monkeypatch, system, s, sem):
    n = 260

    def run():
        return chaos.bif2d(200.0, n, 0.01, s["ic"], s["ranges"], s["idx"], 0, 1e4, 60.0, s["values"], 1, 1e-2,
                           system=system, semantics=sem)
    print(f"bif2d {system} sem={sem} n={n}", flush=True)
    rotating = run()
    # a store for a few hundred wavefronts at a time: ranges that do not rotate
    monkeypatch.setenv("CHAOS_PEAK_STORE_BYTES", str(200 * 64 * 640 * 16))
    assert np.array_equal(rotating, run())
    assert len(np.unique(rotating)) > 3


@pytest.mark.parametrize("sem", [0, 1])
@pytest.mark.parametrize("n", [257, 370])
def test_rotating_basins_equal_served_job(chaos, sem, n):
    ic, vals, rg = [0.0, 0.0, 25.0], [10.0, 24.5, 8 / 3], [-20.0, 20.0, -20.0, 20.0]
    print(f"basins sem={sem} n={n}", flush=True)
    lab, feat, fl = chaos.basins2d(150.0, n, 0.01, ic, rg, [0, 1], 0, 0.0, 110.0, vals, 1, 0.5, system="lorenz_rk4",
                                   semantics=sem)
    srv = chaos.Server()
    job = chaos.make_job(chaos.JOB_BASINS2D, "lorenz_rk4", sem, n, ic, vals, rg, [0, 1], tMax=150.0,
                         transientTime=110.0, eps=0.5)
    jid = srv.submit(job)
    srv.drain()
    lab2, feat2, fl2 = srv.result(jid, job)
    srv.close()
    assert np.array_equal(fl, fl2) and np.array_equal(feat, feat2)
    assert np.array_equal(lab, lab2)


# A transient of negative length is refused by the lane program: the map is 0
# at every size, also where small maps run on lane pairs and larger ones rotate.
@pytest.mark.parametrize("sem", [0, 1])
@pytest.mark.parametrize("n", [1, 5, 128, 200, 260])
def test_negative_transient_gives_a_zero_map_at_every_size(chaos, sem, n):
    print(f"negative transient n={n} sem={sem}", flush=True)
    got = chaos.lle2d(250.0, 0.5, n, 0.01, 1e-7, ROS["ic"], ROS["ranges"], ROS["idx"], -1.0, ROS["values"],
                      system="rossler_rk4", semantics=sem)
    assert np.array_equal(got, np.zeros((n, n)))


# The block size is the caller's choice on every path (plain, lane pairs,
# rotating, rotating pairs) and changes nothing; what was refused is refused.
@pytest.mark.parametrize("n,CT", [(17, 20.0), (60, 250.0), (200, 250.0), (260, 250.0)])
def test_block_option_on_every_exponent_path(chaos, n, CT):
    def run(block):
        print(f"LLE n={n} CT={CT} block={block}", flush=True)
        return chaos.lle2d(CT, 0.5, n, 0.01, 1e-7, ROS["ic"], ROS["ranges"], ROS["idx"], 5.0, ROS["values"],
                           system="rossler_rk4", semantics=1, block=block)
    want = run(0)
    for block in (64, 128, 192, 256):
        assert np.array_equal(run(block), want)
    for block in (32, 100, 320):
        with pytest.raises(Exception):
            run(block)
