"""The sparse prefill's inline-asm quad transposition against the wait states
the compiler does not count around it (CPU test: hipcc builds the translation
unit to gfx950 assembly, nothing runs).

On gfx950 a DPP instruction needs 2 wait states after a VALU write of the
register that it reads from another lane, and an MFMA 2 after a VALU write of
an operand.  The test reads the built code and fails where an inline-asm DPP
move comes too soon after any VALU write of its source, or an MFMA (or a DPP
instruction outside) too soon after a move of the inline asm."""
import os
import re
import subprocess

import pytest

from tests.test_tall_isa import HIPCC, ROOT, _instructions, _regs, _states

SRC = os.path.join(ROOT, "cuda_llm_ops_amd", "csrc", "hip", "sparse_gqa.hip")
STATES = 2


def _operands(t):
    return t.split(None, 1)[1].split(",") if " " in t else []


def _is_dpp(t):
    return "quad_perm" in t or " row_" in t.replace("row_mask", "")


def dpp_hazards(asm):
    insts = _instructions(asm)
    found = []
    for k, (t, a) in enumerate(insts):
        if t.startswith("v_mfma"):
            reads = set().union(*(_regs(o) for o in _operands(t)[1:]))
        elif t.startswith("v_") and _is_dpp(t):
            reads = _regs(_operands(t)[1])   # the DPP operand is the first source
        else:
            continue
        ws = 0
        for t2, a2 in reversed(insts[:k]):
            if ws >= STATES:
                break
            # (between two instructions of the compiler's own it counts them itself)
            if (a or a2) and t2.startswith("v_") and not t2.startswith("v_mfma") and _regs(_operands(t2)[0]) & reads:
                found.append(f"{t2}  ->  {t} after {ws} wait states")
                break
            ws += _states(t2)
    return found


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_sparse_transposition_wait_states(tmp_path):
    out = tmp_path / "sparse.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--cuda-device-only", "-S",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "cuda_llm_ops_amd", "csrc", "hip"),
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", SRC, "-o", str(out)],
                   check=True, capture_output=True, timeout=600)
    asm = out.read_text()
    moves = sum(a and "v_cndmask_b32_dpp" in t for t, a in _instructions(asm))
    assert moves >= 16 and "v_mfma" in asm, "no transposition found: the check would pass vacuously"
    assert moves == 16 * len(re.findall(r";;#ASMSTART\n\s*s_not_b64 vcc", asm))
    found = dpp_hazards(asm)
    assert not found, "\n".join(found[:20])


def test_dpp_scan_finds_planted_cases():
    """The scan itself: a write of a move's source one state before it, a move
    whose source the move before it wrote, and an MFMA one state after the asm
    are reported; the kernel's own pattern is not."""
    bad = """
    v_mov_b32_e32 v1, v9
    ;;#ASMSTART
    s_not_b64 vcc, s[2:3]
    v_cndmask_b32_dpp v5, v1, v2, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf
    v_cndmask_b32_dpp v6, v5, v2, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf
    s_nop 0
    ;;#ASMEND
    v_mfma_f32_16x16x32_bf16 v[20:23], v[4:7], v[8:11], v[20:23]
    """
    assert len(dpp_hazards(bad)) == 3
    good = """
    v_mov_b32_e32 v1, v9
    ;;#ASMSTART
    s_not_b64 vcc, s[2:3]
    s_nop 1
    v_cndmask_b32_dpp v5, v1, v2, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf
    v_cndmask_b32_dpp v7, v3, v2, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf
    s_mov_b64 vcc, s[2:3]
    v_cndmask_b32_dpp v6, v5, v2, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf
    s_nop 1
    ;;#ASMEND
    v_mfma_f32_16x16x32_bf16 v[20:23], v[4:7], v[8:11], v[20:23]
    """
    assert dpp_hazards(good) == []
