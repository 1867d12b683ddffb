"""Register spills of the built stage kernels. A stage kernel that spills
vector registers can be miscompiled (the spill stores of a block may run
before its exec mask is restored, so that lanes reload garbage), so the build
must hold none."""
import os
import re
import subprocess

import pytest

from gocfd_amd import build

LLVM = "/opt/rocm/llvm/bin"


def test_stage_kernels_do_not_spill_vector_registers(tmp_path):
    tools = [os.path.join(LLVM, t) for t in ("llvm-objdump", "llvm-readelf")]
    if not all(os.path.exists(p) for p in tools + [build.LIB]):
        pytest.skip("needs the built library and the ROCm LLVM tools")
    lib = str(tmp_path / "lib.so")
    os.symlink(build.LIB, lib)
    subprocess.run([tools[0], "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    spills = {}
    for f in sorted(tmp_path.iterdir()):
        if build.ARCH not in f.name:
            continue
        notes = subprocess.run([tools[1], "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for k in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", k).group(1)
            spills[name] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", k).group(1))
    stage = {n: s for n, s in spills.items() if re.search(r"k_stage|k_shock|k_prologue|k_halo", n)}
    assert len(stage) > 100
    assert {n: s for n, s in stage.items() if s} == {}
