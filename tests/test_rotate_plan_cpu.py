"""The planning of the rotating launches (rotate_plan.hpp, built by g++): never
more rotating wavefronts than groups, none outside one to eight wavefronts per
SIMD or for short runs; chunks cover a run in at least 12 and at most 48
pieces."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIMDS = 1024


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("rotate") / "rotate_host.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-I", os.path.join(ROOT, "chaoslibrary_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "rotate_host.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    lib.rotate_waves_host.restype = C.c_int
    lib.rotate_waves_host.argtypes = [C.c_int] + [C.c_longlong] * 3
    lib.rotate_chunk_host.restype = C.c_longlong
    lib.rotate_chunk_host.argtypes = [C.c_longlong] * 2
    return lib


@pytest.mark.parametrize("kind", [0, 1])
def test_rotating_wavefronts(lib, kind):
    for groups in list(range(1, 9 * SIMDS, 37)) + [SIMDS, SIMDS + 1, 2 * SIMDS, 8 * SIMDS, 8 * SIMDS + 1]:
        k = lib.rotate_waves_host(kind, groups, SIMDS, 100000)
        assert k in (0, 1, 2) and k * SIMDS <= groups
        if groups <= SIMDS or groups > 8 * SIMDS:
            assert k == 0
        assert lib.rotate_waves_host(kind, groups, SIMDS, 23999) == 0
        assert lib.rotate_waves_host(kind, groups, 0, 100000) == 0
    # one wavefront more than the SIMDs: the case that costs twice at once
    assert lib.rotate_waves_host(kind, SIMDS + 1, SIMDS, 24000) == 1
    # whole numbers of wavefronts per SIMD are even at once
    assert lib.rotate_waves_host(kind, 2 * SIMDS, SIMDS, 10 ** 6) == 0


@pytest.mark.parametrize("unit", [1, 7, 50, 2000, 5000])
def test_chunks(lib, unit):
    rng = np.random.default_rng(unit)
    for ticks in [24000, 24001, 95999, 96000, 96001] + list(rng.integers(24000, 10 ** 9, 200)):
        c = lib.rotate_chunk_host(int(ticks), unit)
        assert c >= 2000 and c % unit == 0
        n = -(-int(ticks) // c)
        assert 1 <= n <= 48
        if unit == 1:
            assert n >= 12
