"""A vector instruction may touch the result of a matrix instruction only some wait states later: 12 after a 32 x 32 x 16
f16 product, 18 after a 32 x 32 x 2 f32 one.  The device does not wait by itself.  The compiler keeps the distance
between its own instructions, but not to those inside asm text: here the built library's instructions are counted,
in the order of the program text."""
import re
import shutil
import subprocess

import pytest

from deers_amd import rocm

OBJDUMP = shutil.which("llvm-objdump") or shutil.which("/opt/rocm/llvm/bin/llvm-objdump")
WAIT_STATES = {"v_mfma_f32_32x32x16_f16": 12, "v_mfma_f32_32x32x2_f32": 18}
OPERAND = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def registers(text):
    out = set()
    for kind, first, last, one in OPERAND.findall(text):
        out |= {(kind, int(one))} if one else {(kind, i) for i in range(int(first), int(last) + 1)}
    return out


def too_early(lines):
    """(kernel, instruction, wait states) of every read or write that comes before a result is there."""
    kernel, pending, found = "", [], []
    for line in lines:
        label = re.match(r"^[0-9a-f]+ <(\w+)>:", line)
        if label:
            kernel, pending = label[1], []
        ins = line.split("//")[0].strip()
        if label or not ins:
            continue
        op = ins.split()[0]
        states = 1 + int(ins.split()[1], 0) if op == "s_nop" else 1
        if op.startswith("v_mfma"):  # accumulators in a chain are forwarded; the other two operands are not
            result, a, b = ins[len(op):].split(", ")[:3]
            touched = registers(a + " " + b)
        elif op.startswith(("v_", "ds_", "global_", "buffer_")):
            result, touched = "", registers(ins)
        else:
            result, touched = "", set()
        found += [(kernel, ins, age) for regs, age, need in pending if age < need and regs & touched]
        pending = [(regs - registers(result), age + states, need) for regs, age, need in pending if age + states < need]
        if op in WAIT_STATES:
            pending.append((registers(result), 0, WAIT_STATES[op]))
        if op in ("s_endpgm", "s_branch"):
            pending = []
    return found


def test_the_count_sees_a_read_that_is_too_early():
    text = ["0 <k>:", "\tv_mfma_f32_32x32x16_f16 v[2:17], v[20:23], v[24:27], 0 // 0", "\ts_nop 5 // 8",
            "\tv_cndmask_b32_e32 v2, v2, v30, vcc // c", "\ts_nop 4", "\tv_add_f32_e32 v0, v17, v0"]
    assert too_early(text) == [("k", "v_cndmask_b32_e32 v2, v2, v30, vcc", 6)]


@pytest.mark.skipif(OBJDUMP is None, reason="needs llvm-objdump")
def test_no_result_of_a_matrix_instruction_is_touched_too_early(tmp_path):
    lib = tmp_path / "lib.so"
    shutil.copy(rocm.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, capture_output=True, cwd=tmp_path)
    objects = sorted(tmp_path.glob("lib.so.*gfx950"))
    assert objects
    seen = 0
    for obj in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True, text=True).stdout
        assert too_early(text.splitlines()) == []
        seen += text.count("v_mfma_f32_32x32")
    assert seen > 1000
