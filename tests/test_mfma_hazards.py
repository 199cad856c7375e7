"""Wait states around the matrix instructions, read off the built library's own code, no GPU.

Some kernels write their matrix instructions as inline assembly (which register file holds what, and in which order things
are issued, decides how they run), and the compiler's hazard pass does not look inside.  What it would have to insert, in
wait states: two between a vector instruction's write of a register and a matrix instruction that reads it; behind a matrix
instruction of n passes (four cycles each) n + 4 (bf16 operands; n + 2: fp32 operands) before anything but the next product of the same sum touches its result: a vector
instruction or a store that reads it, an instruction of either kind that overwrites it, another matrix instruction that takes it as A or B or
as a part of C; and n - 1 before a vector instruction overwrites a C operand that is not the result.
The source keeps these by its order of instructions; a copy that the register allocator puts in between would break them unseen.

Every path is followed from the producer until its wait states have passed: over both sides of a branch, a loop's back edge
and into what comes behind the loop."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "sample_efficient_gpt_amd", "libsegpt_attn.so")
READ_AFTER_VALU = 2
PASSES = {"32x32x16_bf16": 8, "16x16x32_bf16": 4, "32x32x2_f32": 16}
BEHIND_LAST_PASS = {"bf16": 4, "f32": 2}
_REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")
_MEMORY = ("ds_", "global_", "scratch_", "buffer_", "flat_")
_INPUT_ONLY = re.compile(r"ds_write|ds_(add|max|min|or)_|_store|_load_lds_|_atomic")  # no vector register is written (no atomic here returns one)


def _regs(text):
    return frozenset((m[1], i) for m in _REG.finditer(text) for i in range(int(m[2] or m[3]), int(m[2] or m[4]) + 1))


class Instruction:
    def __init__(self, line):
        text, _, comment = line.partition("//")
        self.text = text.strip()
        self.op, _, args = self.text.partition(" ")
        operands = [a.strip() for a in args.split(",")] if args else []
        where = re.match(r"\s*([0-9A-Fa-f]+):", comment)
        self.address = int(where[1], 16) if where else None
        self.passes = self.busy = 0
        if self.op.startswith(("v_mfma", "v_smfma")):
            shape = self.op.split("_", 3)[3]
            self.passes = PASSES[shape]
            self.busy = self.passes + BEHIND_LAST_PASS[shape.split("_")[1]]
        self.is_valu = self.op.startswith("v_") and not self.passes
        self.is_memory = self.op.startswith(_MEMORY)
        written = 0 if self.is_memory and _INPUT_ONLY.search(self.op) else 2 if "swap" in self.op else 1
        self.dst = frozenset().union(*(_regs(o) for o in operands[:written]))
        self.src = _regs(",".join(operands[0 if "swap" in self.op else written:]))
        self.ab = _regs(",".join(operands[1:3])) if self.passes else frozenset()
        self.c = _regs(operands[3]) if self.passes else frozenset()
        self.wait_states = int(operands[0], 0) + 1 if self.op == "s_nop" else 1
        self.target = None  # byte distance behind the next instruction
        if self.op.startswith(("s_cbranch", "s_branch")):
            n = int(operands[0].split()[0], 0)
            self.target = 4 * (n - 65536 if n >= 32768 else n)
        self.goes_on = not self.op.startswith(("s_branch", "s_endpgm", "s_setpc"))


def _conflict(first, then, passed):
    """What is wrong with `then` this many wait states behind `first`, if anything."""
    if first.is_valu:
        return passed < READ_AFTER_VALU and then.passes and first.dst & then.src and "read behind a vector write"
    busy = passed < first.busy
    if busy and (then.is_valu or then.is_memory) and first.dst & then.src:
        return "a result read on its way"
    if busy and (then.is_valu or then.is_memory) and first.dst & then.dst:
        return "a result overwritten on its way"
    if busy and then.passes and first.dst & then.ab:
        return "a result taken as A or B on its way"
    if busy and then.passes and first.dst & then.c and first.dst != then.c:
        return "a result taken as a part of C on its way"
    return passed < first.passes - 1 and then.is_valu and (first.c - first.dst) & then.dst and "C overwritten while it is read"


def violations(lines):
    """Pairs of instructions that are too close on some path."""
    code = [Instruction(l) for l in lines if l.strip() and not l.rstrip().endswith(":") and not l.startswith(("Disassembly", "lib"))]
    code = [i for i in code if i.op and ":" not in i.op]
    at = {i.address: n for n, i in enumerate(code) if i.address is not None}

    def successors(n):
        i = code[n]
        if i.goes_on and n + 1 < len(code):
            yield n + 1
        if i.target is not None:
            yield at[i.address + 4 + i.target]  # a branch is four bytes

    found = []
    for n, first in enumerate(code):
        if not (first.passes or first.is_valu) or not first.dst:
            continue
        limit = first.busy or READ_AFTER_VALU
        seen, todo = {}, [(m, 0) for m in successors(n)]
        while todo:
            m, passed = todo.pop()
            if passed >= limit or seen.get(m, limit) <= passed:
                continue
            seen[m] = passed
            then = code[m]
            what = _conflict(first, then, passed)
            if what:
                found.append((what, first.text, then.text))
            todo += [(k, passed + then.wait_states) for k in successors(m)]
    return found


MFMA = "v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]"
FROM = "v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[4:7], v[32:47]"


@pytest.mark.parametrize("wrong,right", [
    (["v_mov_b32_e32 v5, v9", MFMA], ["v_mov_b32_e32 v8, v9", MFMA]),
    (["v_mov_b32_e32 v5, v9", "s_nop 0", MFMA], ["v_mov_b32_e32 v5, v9", "s_nop 1", MFMA]),
    (["v_swap_b32 v9, v5", MFMA], ["v_swap_b32 v9, v10", MFMA]),
    ([MFMA, "s_nop 10", "v_accvgpr_read_b32 v9, a3"], [MFMA, "s_nop 11", "v_accvgpr_read_b32 v9, a3"]),
    ([MFMA, "s_nop 10", "v_accvgpr_write_b32 a3, v9"], [MFMA, "s_nop 11", "v_accvgpr_write_b32 a3, v9"]),
    ([FROM, "s_nop 10", "scratch_store_dword off, v20, off"], [FROM, "s_nop 11", "scratch_store_dword off, v20, off"]),
    ([FROM, "ds_write_b32 v50, v20"], [FROM, "ds_write_b32 v50, v15"]),
    ([FROM, "ds_read_b128 v[20:23], v50"], [FROM, "ds_read_b128 v[0:3], v50"]),
    ([FROM, "s_nop 5", "v_mov_b32_e32 v40, v9"], [FROM, "s_nop 6", "v_mov_b32_e32 v40, v9"]),
    ([FROM, "s_nop 10", "v_mfma_f32_32x32x16_bf16 v[48:63], v[16:19], v[4:7], v[48:63]"],
     [FROM, "s_nop 11", "v_mfma_f32_32x32x16_bf16 v[48:63], v[16:19], v[4:7], v[48:63]"]),
    ([FROM, "v_mfma_f32_32x32x16_bf16 v[18:33], v[0:3], v[4:7], v[18:33]"], [FROM, "v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[4:7], v[16:31]"]),
    # the loop's next round, then what comes behind the loop
    (["v_mov_b32_e32 v9, v20 // 000000000100: 7E120314", "s_nop 3 // 000000000104: BF800003", FROM + " // 000000000108: D3B70010", "s_cbranch_scc1 65531 // 000000000110: BF85FFFB"],
     ["v_mov_b32_e32 v9, v50 // 000000000100: 7E120332", "s_nop 3 // 000000000104: BF800003", FROM + " // 000000000108: D3B70010", "s_cbranch_scc1 65531 // 000000000110: BF85FFFB"]),
    ([FROM, "s_cbranch_scc1 0 // 000000000110: BF850000", "v_mov_b32_e32 v9, v20 // 000000000114: 7E120314"],
     [FROM, "s_endpgm", "v_mov_b32_e32 v9, v20"]),
])
def test_the_checker_sees_what_it_is_for(wrong, right):
    assert violations(wrong)
    assert not violations(right)


def _code_objects(tmp_path):
    """The library's device code, one file per source, and the path of the LLVM tools."""
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(objdump) or not os.path.exists(LIB):
        pytest.skip("no llvm-objdump, or the library is not built")
    so = shutil.copy(LIB, tmp_path / "lib.so")  # the code objects are written beside the file
    subprocess.run([objdump, "--offloading", str(so)], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    objects = [str(tmp_path / f) for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert objects
    return objects, os.path.dirname(objdump)


def test_built_kernels_keep_the_wait_states(tmp_path):
    objects, tools = _code_objects(tmp_path)
    n_mfma = 0
    for f in objects:
        out = subprocess.run([os.path.join(tools, "llvm-objdump"), "-d", "--mcpu=gfx950", "--no-show-raw-insn", f], check=True, capture_output=True, text=True).stdout
        lines = out.splitlines()
        n_mfma += sum("v_mfma" in l for l in lines)
        found = violations(lines)
        assert not found, (f, len(found), found[:4])
    assert n_mfma > 0


def test_bf16_backward_kernels_keep_everything_in_registers(tmp_path):
    """The bf16 backward loops count their vector-memory operations and are laid out for the registers there are: no scratch."""
    objects, tools = _code_objects(tmp_path)
    seen = {}
    for f in objects:
        notes = subprocess.run([os.path.join(tools, "llvm-readelf"), "--notes", f], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split("  - .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)[1]
            if re.search(r"bwd_(dq|dkdv)_bf16_kernel", name):
                seen[name] = [int(re.search(key + r":\s+(\d+)", kernel)[1]) for key in (r"\.vgpr_spill_count", r"\.private_segment_fixed_size")]
    assert len(seen) >= 16 and all(v == [0, 0] for v in seen.values()), {n: v for n, v in seen.items() if v != [0, 0]}
