"""Wait states around the matrix instructions, read off the built library's own code, no GPU.

Some kernels write their matrix instructions as inline assembly (which register file holds what, and in which order things
are issued, decides how they run), and the compiler's hazard pass does not look inside.  What it would have to insert:
two wait states between a vector instruction's write of a register and a matrix instruction that reads it, and, for the
8-pass 32x32x16 instruction, twelve between its write and a vector instruction that reads or overwrites the result.  The source
keeps both by its order of instructions; a copy that the register allocator puts in between would break them unseen."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "sample_efficient_gpt_amd", "libsegpt_attn.so")
READ_AFTER_VALU, VALU_AFTER_MFMA = 2, 12
_REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")


def _regs(text):
    return {(m[1], i) for m in _REG.finditer(text) for i in range(int(m[2] or m[3]), int(m[2] or m[4]) + 1)}


def violations(lines):
    """Pairs of instructions that are too close, in straight-line order (a branch or its target ends a run)."""
    found, valu, mfma = [], [], []  # (wait states passed since, registers written, text)
    for line in lines:
        text = line.split("//")[0].strip()
        op, _, args = text.partition(" ")
        if not op or text.endswith(":") or op.startswith(("s_cbranch", "s_branch", "s_setpc", "s_endpgm")):
            valu, mfma = [], []
            continue
        operands = [a.strip() for a in args.split(",")]
        is_mfma, is_valu = op.startswith("v_mfma"), op.startswith("v_") and not op.startswith("v_mfma")
        dst = _regs(operands[0]) | (_regs(operands[1]) if "swap" in op and len(operands) > 1 else set())
        src = _regs(",".join(operands[1:]))
        if is_mfma:
            found += [(w, text) for n, r, w in valu if n < READ_AFTER_VALU and r & src]
        if is_valu:
            found += [(w, text) for n, r, w in mfma if n < VALU_AFTER_MFMA and r & (src | dst)]
        passed = int(operands[0], 0) + 1 if op == "s_nop" else 1
        keep = lambda q, limit: [(n + passed, r, w) for n, r, w in q if n + passed < limit]
        valu, mfma = keep(valu, READ_AFTER_VALU), keep(mfma, VALU_AFTER_MFMA)
        if is_mfma:
            mfma.append((0, dst, text))
        elif is_valu:
            valu.append((0, dst, text))
    return found


def test_the_checker_sees_what_it_is_for():
    mfma = "v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]"
    assert violations(["v_mov_b32_e32 v5, v9", mfma])
    assert violations(["v_mov_b32_e32 v5, v9", "s_nop 0", mfma])
    assert not violations(["v_mov_b32_e32 v5, v9", "s_nop 1", mfma])
    assert not violations(["v_mov_b32_e32 v8, v9", mfma])
    assert violations([mfma, "s_nop 10", "v_accvgpr_read_b32 v9, a3"])
    assert not violations([mfma, "s_nop 11", "v_accvgpr_read_b32 v9, a3"])


def test_built_kernels_keep_the_wait_states(tmp_path):
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(objdump) or not os.path.exists(LIB):
        pytest.skip("no llvm-objdump, or the library is not built")
    so = shutil.copy(LIB, tmp_path / "lib.so")  # the code objects are written beside the file
    subprocess.run([objdump, "--offloading", str(so)], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    objects = [f for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert objects
    n_mfma = 0
    for f in objects:
        out = subprocess.run([objdump, "-d", "--mcpu=gfx950", "--no-show-raw-insn", str(tmp_path / f)], check=True, capture_output=True, text=True).stdout
        lines = out.splitlines()
        n_mfma += sum("v_mfma" in l for l in lines)
        assert not violations(lines), (f, violations(lines)[:4])
    assert n_mfma > 0
