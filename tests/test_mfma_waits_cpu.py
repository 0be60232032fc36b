"""Wait states in front of the matrix instructions, in the assembly of the built kernels (no GPU).

A vector instruction's result may be read by a matrix instruction two wait states later at the earliest (an
instruction between them is one, s_nop N is N + 1).  The compiler keeps to that for the instructions that it
knows; it does not see into inline asm.
"""
import os
import re
import subprocess

import pytest

from idi_amd import build as b

KERNELS = ["separable.hip", "adjoint_sep.hip"]
WAIT = 2


def _registers(operand):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.fullmatch(r"v(\d+)", operand)
    return {int(m.group(1))} if m else set()


def unsafe(lines):
    """(line, matrix instruction, writer) wherever a vector write is read too early.  Blocks are taken as they
    follow one another: a wave falls through from one to the next."""
    found, recent, matrix = [], [], 0  # recent: (wait states since, registers, text)
    for number, line in enumerate(lines, 1):
        text = line.split(";")[0].strip()
        if not text or text.endswith(":") or text.startswith("."):
            continue
        name, _, rest = text.partition(" ")
        operands = re.split(r",\s*", rest.strip())
        if name.startswith("v_mfma"):
            matrix += 1
            read = set().union(*(_registers(o.split(" ")[0]) for o in operands[1:4]))
            found += [(number, text, w) for age, regs, w in recent if age < WAIT and regs & read]
        passed = int(operands[0], 0) + 1 if name == "s_nop" else 1
        recent = [(age + passed, regs, w) for age, regs, w in recent if age + passed < WAIT]
        if name.startswith("v_") and not name.startswith("v_mfma"):
            recent.append((0, _registers(operands[0]), text))
            if name.startswith("v_swap"):
                recent.append((0, _registers(operands[1]), text))
    return found, matrix


def test_the_check_sees_a_missing_wait():
    early = ["v_pk_mul_f16 v31, v27, 1.0", "s_waitcnt vmcnt(5)", "v_mfma_f32_16x16x32_f16 v[0:3], v[4:7], v[28:31], 0"]
    assert len(unsafe(early)[0]) == 1
    assert not unsafe([early[0], "s_nop 1", early[2]])[0]
    assert not unsafe(["v_pk_mul_f16 v32, v27, 1.0", early[2]])[0]


@pytest.mark.parametrize("source", KERNELS)
def test_matrix_operands_are_old_enough(source):
    if not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("needs hipcc")
    cmd = [b.hipcc_path(), *b.compile_flags(), *b.FILE_FLAGS.get(source, []), "--cuda-device-only", "-S",
           os.path.join(b.CSRC, source), "-o", "-"]
    out = subprocess.run(cmd, check=True, capture_output=True, text=True).stdout
    found, matrix = unsafe(out.splitlines())
    assert matrix > 50
    assert not found, (len(found), found[:5])
