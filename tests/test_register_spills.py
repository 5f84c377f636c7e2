"""No kernel of the products keeps a vector register in scratch memory, but for the one whose
spill is known and was measured to cost nothing (the plain B X kernel of K >= 768: four values
stored once before the tile loop, reloaded once per tile). The three-part form of that kernel
spilled 19 and ran 8-14% slower than the kernel it replaced, with every result right: nothing
but its time showed it."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"
ALLOWED = {"gemm_bf16_nn16_kernelILi0ELi0ELb0E": 4}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_product_kernels_keep_their_vector_registers(tmp_path):
    asm = tmp_path / "gemm.s"
    cmd = [HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC", "-w", "-mllvm",
           "-pragma-unroll-threshold=1000000", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "--cuda-device-only", "-S",
           os.path.join(ROOT, "dtensor-muon_amd", "csrc", "gemm.hip"), "-o", str(asm)]
    subprocess.run(cmd, check=True, capture_output=True, timeout=900)
    spills = dict(re.findall(r"\.symbol:\s+(\S+)\.kd.*?\.vgpr_spill_count:\s+(\d+)",
                             asm.read_text(), re.S))
    assert sum("nn16" in name for name in spills) == 14 and len(spills) > 40
    over = {name: int(n) for name, n in spills.items()
            if int(n) > next((v for k, v in ALLOWED.items() if k in name), 0)}
    assert not over, over
