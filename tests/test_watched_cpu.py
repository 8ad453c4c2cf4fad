"""A launch that reports an error in its device word fails the call before the
next stage reads its outputs: the call context over a stand-in HIP runtime."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    csrc = os.path.join(ROOT, "chaoslibrary_amd", "csrc")
    so = str(tmp_path_factory.mktemp("watched") / "watched_host.so")
    # -Bsymbolic: the stand-ins are found before a HIP runtime in the process
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-fPIC", "-shared", "-Wl,-Bsymbolic",
                    "-I", csrc, "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "native", "watched_host.cpp"),
                    os.path.join(csrc, "runtime.cpp"), "-o", so], check=True, capture_output=True)
    lib = C.CDLL(so)
    lib.watched_call.restype = C.c_int
    lib.watched_call.argtypes = [C.c_int]
    return lib


def test_error_word_stops_the_call_before_its_outputs_are_read(lib):
    assert lib.watched_call(0) == 1
    assert lib.watched_call(1) == 2
    assert lib.watched_call(-5) == 2
