"""Places of a peak chunk's entries before they are scattered: a permutation in
order of (lane, sequence) for a chunk that its wave filled, and never outside
the chunk whatever the words hold (sequence numbers that repeat, wrap or leave
gaps)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    so = str(tmp_path_factory.mktemp("place") / "chunk_place_host.so")
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-I", os.path.join(ROOT, "chaoslibrary_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "native", "chunk_place_host.cpp"), "-o", so],
                   check=True, capture_output=True)
    return C.CDLL(so)


def places(lib, kl):
    out = np.zeros(kl.size, dtype=np.int32)
    lib.chunk_places(kl.ctypes.data_as(C.c_void_p), C.c_int(kl.size), out.ctypes.data_as(C.c_void_p))
    return out


@pytest.mark.parametrize("n", [1, 2, 63, 64, 255, 256])
def test_filled_chunk_is_put_in_order(lib, n):
    rng = np.random.default_rng(n)
    nxt = rng.integers(0, 1 << 25, 64)
    kl = np.zeros(n, dtype=np.uint32)
    for s, lane in enumerate(rng.integers(0, 64, n)):
        kl[s] = (int(nxt[lane]) << 6) | int(lane)
        nxt[lane] += 1
    got = places(lib, kl)
    want = np.argsort(np.lexsort((kl >> 6, kl & 63)))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("kind", ["any", "gaps", "repeats", "wrap", "zero"])
def test_places_stay_inside_the_chunk(lib, kind):
    rng = np.random.default_rng(7)
    for n in (1, 64, 256):
        lane = rng.integers(0, 64, n)
        seq = {"any": rng.integers(0, 1 << 26, n), "gaps": 3 * np.arange(n), "repeats": np.arange(n) // 5,
               "wrap": (np.arange(n) - 100) % (1 << 26), "zero": np.zeros(n, dtype=int)}[kind]
        kl = ((seq.astype(np.uint64) << np.uint64(6)) | lane.astype(np.uint64)).astype(np.uint32)
        got = places(lib, kl)
        assert got.min() >= -1 and got.max() < n
