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


def test_asm_loads_bring_their_wait_states(functions):
    loads = 0
    for name, lines in functions.items():
        states = last = 0
        for block, op, args in lines:
            if block != last:
                states, last = 0, block  # what came before the block may have written its operands
            if not block:
                continue
            if op.startswith(("buffer_", "global_", "scratch_", "flat_")):
                loads += 1
                assert states >= SGPR_READ_STATES, (name, op, args, states)
            states += _states(op, args)
    assert loads > 0


def test_asm_blocks_have_m0_to_themselves(functions):
    """A block sets m0 for its own load; kernels with such blocks use it nowhere else."""
    kernels = 0
    for name, lines in functions.items():
        users = [bool(block) for block, _, args in lines if re.search(r"\bm0\b", args)]
        if any(users):
            kernels += 1
            assert all(users), name
    assert kernels > 0
