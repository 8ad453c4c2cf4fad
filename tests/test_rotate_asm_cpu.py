"""Active lanes in the built code: the rotating kernels check that a wavefront's
64 lanes are together where it takes a ticket (rotate.hpp), and the sweeps'
masked moves (lanes.hpp) do not assume which lanes are active."""
import os
import re

import pytest

from test_build_guard import BUILD, LLVM, _device_asm


@pytest.mark.parametrize("obj,kernels", [("lle.o", ["lle_rotate_kernel", "lle_pair_rotate_kernel"]),
                                         ("sweep_rotate.o", ["sweep_rotate_kernel"])])
def test_rotating_kernels_check_for_whole_wavefronts(tmp_path, obj, kernels):
    path = os.path.join(BUILD, obj)
    if not os.path.exists(path) or not os.path.exists(f"{LLVM}/llvm-objdump"):
        pytest.skip("no built objects or no ROCm LLVM tools")
    asm = _device_asm(path, str(tmp_path))
    bodies = re.split(r"\n[0-9a-f]+ <(\w+)>:\n", asm)[1:]
    for kernel in kernels:
        found = [(n, b) for n, b in zip(bodies[::2], bodies[1::2]) if kernel in n]
        assert len(found) >= 7
        for name, body in found:
            assert re.search(r"\bs_cmp_(eq|lg)_u64 exec, -1\b", body), name


# The sweeps move pending peaks under a lane mask written to exec; the lanes
# that were active come back from a saved copy, not from "all 64".
@pytest.mark.parametrize("obj", ["sweep.o", "sweep_rotate.o", "engine.o"])
def test_sweeps_restore_the_active_lanes_they_had(tmp_path, obj):
    path = os.path.join(BUILD, obj)
    if not os.path.exists(path) or not os.path.exists(f"{LLVM}/llvm-objdump"):
        pytest.skip("no built objects or no ROCm LLVM tools")
    asm = _device_asm(path, str(tmp_path))
    assert not re.search(r"\bs_mov_b64 exec, -1\b", asm)
