"""Wait states around inline assembly.  A vector-memory instruction may read a scalar register no sooner than five wait states after a vector
instruction wrote it (v_readlane, v_readfirstlane, compares).  The compiler keeps that distance for instructions of its own; it does not look
into asm statements.  Runs without a GPU."""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNELS = os.path.join(ROOT, "flux_amd", "csrc", "kernels")
OBJECTS = sorted(glob.glob(os.path.join(ROOT, "flux_amd", "lib", "obj", "*.o")))
OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")) if p and os.path.exists(p)), None)
WAIT_STATES = 5
MEMORY = ("buffer_", "global_", "flat_", "scratch_")


def wait_states(instruction):
    return int(instruction.split()[1], 0) + 1 if instruction.startswith("s_nop") else 1


def test_asm_statements_that_set_up_their_loads_wait_themselves():
    """Statements of several instructions with a load: whatever the compiler puts in front, the first load is far enough from it."""
    seen = 0
    for path in sorted(glob.glob(os.path.join(KERNELS, "*.h*"))):
        for statement in re.findall(r"asm volatile\((.*?)\)\s*;", open(path).read(), re.S):
            text = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', re.split(r'"\s*(?:\\\n\s*)?:', statement)[0] + '"'))
            lines = [i.strip() for i in text.replace("\\t", " ").split("\\n") if i.strip()]
            loads = [n for n, i in enumerate(lines) if i.startswith(MEMORY)]
            if not loads or len(lines) == 1:
                continue
            seen += 1
            before = sum(wait_states(i) for i in lines[:loads[0]])
            assert before >= WAIT_STATES, f"{os.path.basename(path)}: {lines[:loads[0] + 1]}"
    assert seen >= 2


REGISTERS = re.compile(r"\bs(\d+)\b|\bs\[(\d+):(\d+)\]|\b(vcc|m0)\b")


def scalars(operands):
    out = set()
    for one, first, last, name in REGISTERS.findall(operands):
        out |= {int(one)} if one else set(range(int(first), int(last) + 1)) if first else {name}
    return out


def too_close(lines):
    """Loads and stores, in layout order, that read a scalar register a vector instruction wrote less than five wait states before."""
    kernel, now, written, found = "", 0, {}, []
    for line in lines:
        if line.endswith(">:\n"):
            kernel, written = line.split("<")[-1][:-3], {}
        elif line.startswith("\t"):
            instruction = line.split("//")[0].strip()
            op, _, operands = instruction.partition(" ")
            if op.startswith(MEMORY):
                found += [f"{kernel}: {instruction}" for r in scalars(operands) if now - written.get(r, -WAIT_STATES - 1) - 1 < WAIT_STATES]
            elif op.startswith("v_"):
                for r in scalars(",".join(operands.split(",")[:2 if "_co_" in op or op.startswith(("v_div_scale", "v_mad_u64", "v_mad_i64")) else 1])):
                    written[r] = now
            elif op.startswith("s_") and not op.startswith(("s_cmp", "s_bitcmp", "s_nop")):
                for r in scalars(operands.split(",")[0]):
                    written.pop(r, None)
            now += wait_states(instruction)
    return found


def test_the_scan_sees_a_load_that_is_too_close():
    code = ["0 <k>:\n", "\tv_readlane_b32 s5, v1, 3\n", "\ts_mov_b32 m0, s9\n", "\ts_nop 0\n", "\tbuffer_load_dwordx4 v2, s[4:7], s8 offen lds\n"]
    assert len(too_close(code)) == 1
    assert too_close(code[:3] + ["\ts_nop 3\n"] + code[4:]) == []
    assert too_close(code[:2] + ["\ts_mov_b32 s5, s9\n"] + code[2:]) == []


@pytest.mark.skipif(OBJDUMP is None or not OBJECTS, reason="needs llvm-objdump and built objects")
@pytest.mark.parametrize("obj", OBJECTS, ids=[os.path.basename(o) for o in OBJECTS])
def test_built_kernels_keep_the_distance(obj, tmp_path):
    """All kernels as built: their asm statements of a single load rely on what the compiler puts around them."""
    copy = shutil.copy(obj, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, capture_output=True)
    for code in glob.glob(copy + ".*gfx950"):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", code], check=True, capture_output=True, text=True).stdout
        assert too_close(text.splitlines(True)) == []
