"""The wave peak detector's mask logic (PeakMasks in
chaoslibrary_amd/csrc/peaks.hpp, built for the host) against the oracle's
peakFinder on rows with plateaus that fall, rise again and reach the end,
steps of the order of the 1e-13 threshold, flat rows and NaN / infinite tails;
the sweeps' shortcut over samples that need no work changes nothing."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import _oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_D, _I = C.POINTER(C.c_double), C.POINTER(C.c_int)


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    so = str(tmp_path_factory.mktemp("peakmasks") / "peak_masks_host.so")
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-ffp-contract=off", "-I", os.path.join(ROOT, "chaoslibrary_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "native", "peak_masks_host.cpp"),
                    "-o", so], check=True, capture_output=True)
    lib = C.CDLL(so)
    lib.host_peak_masks.restype = None
    lib.host_peak_masks.argtypes = [_D, C.c_int, C.c_int, _I, _D, _I]
    return lib


def rows(kind, n, rng):
    if kind == "steps":       # small integers: long plateaus, rises out of them
        return np.cumsum(rng.integers(-1, 2, (64, n)), axis=1).astype(float)
    if kind == "threshold":   # steps around 1e-13
        return np.cumsum(rng.choice([-2e-13, -1e-13, -0.4e-13, 0.0, 0.4e-13, 1e-13, 2e-13], (64, n)), axis=1)
    if kind == "smooth":      # rarely an event in any row
        ph = rng.uniform(0, 6.3, (64, 1))
        return np.sin(ph + np.arange(n) * rng.uniform(0.001, 0.05, (64, 1)))
    d = np.cumsum(rng.integers(-1, 2, (64, n)), axis=1).astype(float)
    cut = rng.integers(0, n + 1, 64)
    for l in range(64):       # diverged tails and constant rows
        d[l, cut[l]:] = [np.nan, np.inf, -np.inf, 3.0][l % 4]
    return d


@pytest.mark.parametrize("kind", ["steps", "threshold", "smooth", "tails"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 64, 501])
def test_masks_equal_reference_peak_finder(host, kind, n):
    rng = np.random.default_rng(n)
    for rep in range(6):
        d = np.ascontiguousarray(rows(kind, n, rng))
        got = []
        for shortcut in (0, 1):
            counts = np.zeros(64, dtype=np.int32)
            values, times = np.zeros((64, n)), np.zeros((64, n), dtype=np.int32)
            with np.errstate(invalid="ignore"):
                host.host_peak_masks(d.ctypes.data_as(_D), n, shortcut, counts.ctypes.data_as(_I),
                                     values.ctypes.data_as(_D), times.ctypes.data_as(_I))
            got.append((counts, values, times))
        for a, b in zip(*got):
            assert np.array_equal(a, b)
        counts, values, times = got[0]
        for l in range(64):
            # the reference drops the first peak; intervals are time differences
            pk, iv = O.peak_finder(d[l], 0.5)
            k = max(0, counts[l] - 1)
            assert k == pk.size
            assert np.array_equal(values[l, 1:counts[l]], pk[:k])
            assert np.array_equal(np.diff(times[l, :counts[l]]) * 0.5 if counts[l] else np.zeros(0), iv[:k])
