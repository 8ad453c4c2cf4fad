"""The sweeps' pairs of samples (SamplePair, peaks.hpp, built for the host)
against the oracle's peakFinder on each lane's samples up to its divergence:
peaks that wait in a slot, second peaks of a lane, plateaus and values outside
the divergence band in either half of a pair.  Lanes that no longer integrate
cost the others nothing."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import _oracle as O
from test_peak_masks_cpu import rows

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_D, _I = C.POINTER(C.c_double), C.POINTER(C.c_int)


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    so = str(tmp_path_factory.mktemp("pairs") / "sample_pairs_host.so")
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-ffp-contract=off", "-I", os.path.join(ROOT, "chaoslibrary_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "native", "sample_pairs_host.cpp"),
                    "-o", so], check=True, capture_output=True)
    lib = C.CDLL(so)
    lib.host_sample_pairs.restype = C.c_int
    lib.host_sample_pairs.argtypes = [_D, C.c_int, C.c_double, C.c_double, _I, _D, _I]
    return lib


def run(host, d, bound, band):
    d = np.ascontiguousarray(d)
    n = d.shape[1]
    counts = np.zeros(64, dtype=np.int32)
    values, times = np.zeros((64, n)), np.zeros((64, n), dtype=np.int32)
    with np.errstate(invalid="ignore"):
        slow = host.host_sample_pairs(d.ctypes.data_as(_D), n, bound, band, counts.ctypes.data_as(_I),
                                      values.ctypes.data_as(_D), times.ctypes.data_as(_I))
    return slow, counts, values, times


@pytest.mark.parametrize("kind", ["steps", "threshold", "smooth", "tails"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 64, 501])
@pytest.mark.parametrize("bound", [np.inf, 6.0, 0.9])
def test_pairs_equal_reference_peak_finder(host, kind, n, bound):
    rng = np.random.default_rng(n)
    for rep in range(4):
        d = rows(kind, n, rng)
        _, counts, values, times = run(host, d, bound, bound if np.isfinite(bound) else 1e300)
        for lane in range(64):
            out = np.nonzero(~np.isfinite(d[lane]) | (np.abs(d[lane]) > bound))[0]
            # a peak needs the sample after it, tested for divergence first
            pk, iv = O.peak_finder(d[lane, :out[0]] if out.size else d[lane], 0.5)
            k = max(0, counts[lane] - 1)
            assert k == pk.size
            assert np.array_equal(values[lane, 1:counts[lane]], pk[:k])
            assert np.array_equal(np.diff(times[lane, :counts[lane]]) * 0.5 if counts[lane] else np.zeros(0), iv[:k])


# A lane that left the band on its way up and then stays where it is holds an
# open plateau to the end of the record.
def test_a_stopped_lane_does_not_slow_the_others(host):
    n = 4001
    d = np.sin(np.arange(64)[:, None] + 0.01 * np.arange(n))
    d[0] = np.minimum(np.arange(n) * 0.5, 40.0)
    slow, *_ = run(host, d, 2.0, 2.0)
    d[0] = d[1]
    base, *_ = run(host, d, 2.0, 2.0)
    assert slow <= base + 2
