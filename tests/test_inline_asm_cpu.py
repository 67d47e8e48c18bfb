"""The loads that the attention kernels issue from inline asm, in the assembly that the compiler
makes of them.  It inserts no wait states for instructions of an asm block and follows no register
that a block writes without saying so, so each block has to be right by itself."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from compactattention_amd import build

SGPR_READ_STATES = 5  # wait states from a vector instruction that writes an SGPR to a memory instruction that reads it


def _states(op, args):
    """Wait states that an instruction is worth to one after it."""
    return int(args.split()[0], 0) + 1 if op == "s_nop" else 1


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    """name -> lines of (asm block number or 0, opcode, operands) of every kernel of ca_attn.hip."""
    out = str(tmp_path_factory.mktemp("asm") / "attn.s")
    flags = [a for a in build.command(out) if not a.endswith(".hip") and a not in ("-shared", "-o", out)]
    subprocess.run(flags + ["-S", "--cuda-device-only", "-o", out, os.path.join(build.CSRC, "ca_attn.hip")], check=True,
                   capture_output=True)
    found, lines, block, blocks = {}, None, 0, 0
    for text in open(out):
        label = re.match(r"(_Z\w+):", text)
        if label:
            lines, block = found.setdefault(label[1], []), 0
        if ";;#ASMSTART" in text:
            blocks += 1
            block = blocks
        elif ";;#ASMEND" in text:
            block = 0
        code = text.split(";")[0].strip()
        if lines is None or not code or code.startswith(".") or code.endswith(":"):
            continue
        op, _, args = code.partition(" ") if " " in code else code.partition("\t")
        lines.append((block, op, args.strip()))
    return found


def _sgprs(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]|s(\d+)", operand)
    return set() if m is None else {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))


def _vector_writes(op, args):
    """SGPRs that a vector instruction may write (the first operand, or the second of those with a carry)."""
    operands = [a.split()[0] for a in args.split(",")] if op.startswith("v_") else []
    return set().union(*(_sgprs(a) for a in operands[:1 if re.match("v_read", op) else 2]))


def test_asm_loads_have_their_wait_states(functions):
    """Five wait states lie between a vector write of a load's SGPRs and the load: in its own asm block,
    or the kernel waits them once ("s_nop 4") and no vector instruction writes those SGPRs from there on."""
    whole, fixed = 0, 0
    for name, lines in functions.items():
        loads, settled = [], None
        states = last = 0
        for i, (block, op, args) in enumerate(lines):
            if block != last:
                states, last = 0, block  # what came before the block may have written its operands
            if not block:
                continue
            if (op, args) == ("s_nop", str(SGPR_READ_STATES - 1)):
                settled = i
            if op.startswith(("buffer_", "global_", "scratch_", "flat_")):
                loads.append((i, states, set().union(*(_sgprs(a.split()[0]) for a in args.split(",")))))
            states += _states(op, args)
        for i, states, read in loads:
            if states >= SGPR_READ_STATES:
                whole += 1
                continue
            fixed += 1
            assert settled is not None and settled < i, (name, i, states)
            for block, op, args in lines[settled + 1:loads[-1][0]]:
                assert not read & _vector_writes(op, args), (name, op, args)
    assert whole > 0 and fixed > 0


def test_asm_blocks_have_m0_to_themselves(functions):
    """A block sets m0 for its own load; kernels with such blocks use it nowhere else."""
    kernels = 0
    for name, lines in functions.items():
        users = [bool(block) for block, _, args in lines if re.search(r"\bm0\b", args)]
        if any(users):
            kernels += 1
            assert all(users), name
    assert kernels > 0
