"""Distances around the matrix instructions that the prompt kernel writes out, in the built library's gfx950 code.

The compiler keeps the required distances around its own matrix instructions, but does not look into inline assembly.  What it
keeps for v_mfma_f32_16x16x32_f16 on gfx950: two instructions (or s_nop 1) between a vector instruction's result and the
product that reads it, eight between a product's result and another instruction that touches it, none between products that add to
the same accumulator.  Checked along straight code: labels are passed over."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mixed-precision-cuda-kernel_amd", "libcherryq.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def registers(operand):
    m = re.fullmatch(r"[-|]*([va])\[(\d+):(\d+)\]\|?", operand) or re.fullmatch(r"[-|]*([va])((\d+))\|?", operand)
    return {(m[1], i) for i in range(int(m[2]), int(m[3]) + 1)} if m else set()


def waits(op, operands):
    return int(operands[0], 0) + 1 if op == "s_nop" else 1


def too_close(instructions):
    """[(what, distance, instruction)] of a kernel's [(opcode, [operands])]"""
    found = []
    for i, (op, operands) in enumerate(instructions):
        if not op.startswith("v_mfma"):
            continue
        out, read = registers(operands[0]), set().union(*map(registers, operands[1:4]))
        gap, j = 0, i - 1
        while j >= 0 and gap < 2:
            o, x = instructions[j]
            if o.startswith("v_") and not o.startswith(("v_mfma", "v_cmp", "v_readfirstlane", "v_nop")) and x and registers(x[0]) & read:
                found.append(("vector result -> product", gap, (o, x)))
            gap, j = gap + waits(o, x), j - 1
        gap, j = 0, i + 1
        while j < len(instructions) and gap < 8:
            o, x = instructions[j]
            touched = set().union(set(), *map(registers, x))
            if o.startswith("v_mfma"):
                if registers(x[0]) & out and registers(x[0]) != out or (registers(x[1]) | registers(x[2])) & out:
                    found.append(("product -> other product", gap, (o, x)))
                if registers(x[0]) == out:
                    break
            elif touched & out:
                found.append(("product -> instruction", gap, (o, x)))
                break
            gap, j = gap + waits(o, x), j + 1
    return found


def test_the_check_finds_what_is_too_close():
    mfma = ("v_mfma_f32_16x16x32_f16", ["v[0:3]", "v[8:11]", "v[12:15]", "v[0:3]"])
    mov, nop = ("v_mov_b32_e32", ["v9", "0"]), ("s_nop", ["1"])
    assert too_close([mov, mfma]) and too_close([mov, ("s_nop", ["0"]), mfma]) and not too_close([mov, nop, mfma])
    reader = ("v_add_f32_e32", ["v20", "v3", "v4"])
    assert too_close([mfma, reader]) and too_close([mfma, ("s_nop", ["6"]), reader]) and not too_close([mfma, ("s_nop", ["7"]), reader])
    assert not too_close([mfma, mfma]) and too_close([mfma, ("v_mfma_f32_16x16x32_f16", ["v[4:7]", "v[0:3]", "v[12:15]", "v[4:7]"])])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs ROCm's llvm-objdump")
def test_prompt_kernels_keep_their_distances(tmp_path):
    assert os.path.exists(LIB), "build the library first (python mixed-precision-cuda-kernel_amd/build.py)"
    lib = shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    kernels = {}
    for name in sorted(os.listdir(tmp_path)):
        path = str(tmp_path / name)
        if not name.endswith("gfx950") or b"prompt_shared_k_kernel" not in open(path, "rb").read():
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", path], check=True, capture_output=True,
                              text=True).stdout
        for symbol, body in re.findall(r"^<(\S*prompt_\w*kernel\S*)>:\n(.*?)(?=^<|\Z)", text, re.S | re.M):
            code = [line.split("//")[0].split(None, 1) for line in body.splitlines() if line.strip() and not line.rstrip().endswith(":")]
            kernels[symbol] = [(x[0], [o.strip() for o in x[1].split(",")] if len(x) > 1 else []) for x in code if x]
    products = {symbol: code for symbol, code in kernels.items() if any(op.startswith("v_mfma") for op, _ in code)}
    assert len(products) >= 52
    for symbol, code in products.items():
        assert not too_close(code), (symbol, too_close(code)[:4])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs ROCm's llvm-objdump")
def test_every_prompt_kernel_is_among_those_checked(tmp_path):
    """One kernel a line of the shape tables, both widths of codes, groups of whole units and others: all of them by the names that the test
    above looks for, with matrix instructions inside."""
    lib = shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    products = 0
    for name in sorted(os.listdir(tmp_path)):
        path = str(tmp_path / name)
        if name.endswith("gfx950") and b"prompt_shared_k_kernel" in open(path, "rb").read():
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", path], check=True, capture_output=True,
                                  text=True).stdout
            bodies = re.findall(r"^<\S*prompt_\w*kernel\S*>:\n(.*?)(?=^<|\Z)", text, re.S | re.M)
            products += sum("v_mfma" in body for body in bodies)
    source = open(os.path.join(os.path.dirname(LIB), "csrc", "cq_prompt.hip")).read()
    shapes = len(re.findall(r"^    X\(\d+,", source, re.M))
    assert shapes >= 15 and products == 4 * shapes
