"""The dK/dV kernel's inline-asm MFMAs against the wait states the compiler
does not count for them (CPU test: hipcc builds the translation unit to gfx950
assembly, nothing runs), with the scan of the tall prefill's test: no access to
an accumulator within 24 wait states of the MFMA that wrote it, and no VALU
write of an operand within the 2 states before one."""
import os
import re
import subprocess

import pytest

from tests.test_tall_isa import HIPCC, ROOT, hazards

SRC = os.path.join(ROOT, "cuda_llm_ops_amd", "csrc", "hip", "flash_gqa_backward_dkdv.hip")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_dkdv_inline_mfma_wait_states(tmp_path):
    out = tmp_path / "dkdv.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--cuda-device-only", "-S",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "cuda_llm_ops_amd", "csrc", "hip"),
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-mllvm", "-amdgpu-mfma-vgpr-form", SRC, "-o", str(out)],
                   check=True, capture_output=True, timeout=600)
    asm = out.read_text()
    assert re.search(r";;#ASMSTART\n\s*v_mfma", asm), "no inline-asm MFMA found: the check would pass vacuously"
    found = hazards(asm)
    assert not found, "\n".join(found[:20])
