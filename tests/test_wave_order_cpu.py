"""Lanes of a wave that hand values to each other through LDS without a workgroup barrier: the order of the
writes and reads stands in the code's LLVM IR, and does not hang on what the compiler can tell apart (no GPU)."""
import os
import subprocess

import pytest

from idi_amd import build as b


@pytest.mark.parametrize("source,kernel", [("correlate.hip", "k_qcorr_runs")])
def test_wave_barriers_order_memory(source, kernel):
    if not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("needs hipcc")
    cmd = [b.hipcc_path(), *b.compile_flags(), "--cuda-device-only", "-S", "-emit-llvm", os.path.join(b.CSRC, source),
           "-o", "-"]
    text = subprocess.run(cmd, check=True, capture_output=True, text=True).stdout
    text = next(f for f in text.split("\ndefine ")[1:] if kernel in f.split("\n", 1)[0])
    lines = [s.strip() for s in text[:text.index("\n}\n")].splitlines()]
    at = [i for i, s in enumerate(lines) if "@llvm.amdgcn.wave.barrier" in s]
    assert at
    for i in at:
        assert lines[i - 1] == 'fence syncscope("wavefront") release', lines[i - 3:i]
        assert lines[i + 1] == 'fence syncscope("wavefront") acquire', lines[i:i + 3]
