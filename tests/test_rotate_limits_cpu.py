"""Limits of the rotating launches' plan (rotate_plan.hpp, built by g++): a
chunk is short enough to be waited for, and the tickets stay countable, however
long the run, its windows and its samples are."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIMDS = 1024
# a waiting wavefront polls 2^27 times with a sleep of 1024 clocks at 2.4 GHz
# between, 57 s or more; a step takes at most 4 us
CHUNK_STEPS = 57 / 4e-6 / 4


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("limits") / "rotate_limits_host.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-I", os.path.join(ROOT, "chaoslibrary_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "rotate_limits_host.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    lib.plan_waves.restype = C.c_int
    lib.plan_waves.argtypes = [C.c_int] + [C.c_longlong] * 5
    lib.plan_chunk.restype = C.c_longlong
    lib.plan_chunk.argtypes = [C.c_longlong] * 3
    return lib


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("groups", [1025, 1407, 2600, 5600, 8000])
def test_chunks_can_be_waited_for(lib, kind, groups):
    rng = np.random.default_rng(groups)
    for steps in (1, 2, 3, 100, 10 ** 4, 10 ** 7, 2 ** 31 - 1):
        for unit in (1, 50, 40000, 10 ** 7):
            for ticks in [24000, 10 ** 6, 2 ** 31, 2 ** 32] + [int(10.0 ** e) for e in rng.uniform(4.4, 9.6, 20)]:
                if lib.plan_waves(kind, groups, SIMDS, ticks, unit, steps) == 0:
                    continue
                chunk = lib.plan_chunk(ticks, unit, steps)
                assert chunk >= 1 and chunk % unit == 0
                assert chunk * steps <= CHUNK_STEPS
                assert -(-ticks // chunk) * groups < 1 << 25


# runs longer than the plan can cut keep the plain launch; long ones it can cut
# still rotate
def test_long_runs_keep_a_plan(lib):
    assert lib.plan_waves(0, 1407, SIMDS, 2 ** 32, 1, 2) == 1
    assert lib.plan_waves(0, 1407, SIMDS, 2 ** 31, 50, 1) == 1
    assert lib.plan_waves(1, 1407, SIMDS, 2 ** 31, 1, 1) == 1
    assert lib.plan_waves(1, 1407, SIMDS, 2 ** 31, 1, 10 ** 6) == 0


# Few chunks, of one long window each: taken in turns only where the whole
# rounds they need are fewer than the wavefronts of the fullest SIMD.
@pytest.mark.parametrize("groups", [1025, 1250, 1407, 1800, 2047])
def test_few_long_chunks_count_whole_rounds(lib, groups):
    unit = 40000
    for windows in range(1, 12):
        rounds = -(-groups * windows // SIMDS)
        got = lib.plan_waves(0, groups, SIMDS, windows * unit, unit, 1)
        assert got == (1 if 1.03 * rounds / windows < 0.98 * 2 else 0), windows
    assert lib.plan_waves(0, groups, SIMDS, unit, unit, 1) == 0
