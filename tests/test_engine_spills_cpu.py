"""The engine's persistent kernels run at a register cap chosen for their
wavefronts per SIMD; none of them spills a vector register to memory."""
import os
import re
import subprocess

import pytest

from test_build_guard import BUILD, LLVM, TARGET


def test_engine_kernels_spill_no_vector_registers(tmp_path):
    obj = os.path.join(BUILD, "engine.o")
    if not os.path.exists(obj) or not os.path.exists(f"{LLVM}/llvm-readelf"):
        pytest.skip("no built objects or no ROCm LLVM tools")
    fb, co = str(tmp_path / "engine.fb"), str(tmp_path / "engine.co")
    subprocess.run([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fb}", obj, str(tmp_path / "engine.o")],
                   check=True)
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={fb}",
                    f"--targets={TARGET}", f"--output={co}"], check=True)
    notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", co], check=True, capture_output=True, text=True).stdout
    spills = {}
    for k in re.split(r"\n  - ", notes)[1:]:
        name, count = re.search(r"\.name:\s+(\S+)", k), re.search(r"\.vgpr_spill_count:\s+(\d+)", k)
        if name and count:
            spills[name.group(1)] = int(count.group(1))
    engine = {n: c for n, c in spills.items() if "engine_" in n}
    assert len(engine) == 20  # two exponent families, eighteen sweep families
    assert not any(engine.values()), {n: c for n, c in engine.items() if c}
