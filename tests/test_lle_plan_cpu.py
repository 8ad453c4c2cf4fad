"""Which kernel an exponent map gets (rotate_plan.hpp, built by g++)."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIMDS = 1024


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("lleplan") / "lle_plan_host.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-I", os.path.join(ROOT, "chaoslibrary_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "lle_plan_host.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    for f in (lib.lle_split_host, lib.lle_turn_host):
        f.restype = C.c_int
        f.argtypes = [C.c_longlong] * 5
    return lib


# The lane pairs and the rotating kernels do not ask LleProg::ticks whether a
# run may start, so a run that it refuses must not reach them.
@pytest.mark.parametrize("groups", [1, 300, 900, 1025, 1407, 2500])
def test_a_refused_run_keeps_the_plain_kernel(lib, groups):
    for S in (-1, -100, -2 ** 31):
        assert not lib.lle_split_host(groups, SIMDS, S, 1000, 50)
        assert not lib.lle_turn_host(groups, SIMDS, S, 1000, 50)
    assert lib.lle_split_host(groups, SIMDS, 0, 1000, 50) == (groups <= 900)
    assert (lib.lle_turn_host(groups, SIMDS, 0, 1000, 50) > 0) == (groups > SIMDS)


# Lane pairs double the work of a window's end: above one wavefront of pairs a
# SIMD they are taken only where turns make up for it, so neither for windows of
# a few steps nor for runs too short for turns.
def test_short_windows_and_short_runs_stay_on_one_lane(lib):
    for groups in (520, 625, 900):
        for NTp in (1, 2, 4, 8, 16, 50, 100):
            assert not lib.lle_split_host(groups, SIMDS, 500, 20000 // NTp, NTp)
    assert not lib.lle_split_host(625, SIMDS, 500, 40000, 1)
    assert lib.lle_split_host(625, SIMDS, 500, 800, 50)
    for groups in (1, 100, 512):
        for NTp in (1, 50):
            assert lib.lle_split_host(groups, SIMDS, 500, 200 // NTp, NTp)
            assert not lib.lle_split_host(groups, SIMDS, 500, 199 // NTp, NTp)
