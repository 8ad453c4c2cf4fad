"""chaos_options.block in the rotating launches of the exponent maps: blocks of
any size that the option takes hold the wavefronts that the plan asked for."""
import ctypes as C
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("blocks") / "rotate_blocks_host.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-I", os.path.join(ROOT, "chaoslibrary_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "rotate_blocks_host.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    lib.blocks_host.restype = C.c_uint
    lib.blocks_host.argtypes = [C.c_longlong, C.c_int, C.c_int]
    return lib


@pytest.mark.parametrize("block", [64, 128, 192, 256])
@pytest.mark.parametrize("waves", [1, 2])
@pytest.mark.parametrize("cus", [1, 32, 256])
def test_blocks_hold_the_planned_wavefronts(lib, cus, waves, block):
    n = lib.blocks_host(cus, waves, block) * (block // 64)
    assert 0 <= n - 4 * cus * waves < block // 64


def test_every_exponent_map_kernel_is_launched_with_the_option():
    src = open(os.path.join(ROOT, "chaoslibrary_amd", "csrc", "lle.hip")).read()
    launches = re.findall(r"hipLaunchKernelGGL\((\w+)<S>, dim3\(.*?\), dim3\((\w+)\)", src, re.S)
    assert len(launches) == 5
    assert all(block == "block" for _, block in launches), launches
