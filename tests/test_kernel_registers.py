"""Kernels whose speed rests on how many of their waves a SIMD holds: their registers, from the device code's own notes.  A
SIMD has 512 registers a lane and hands them out to a wave in eights, so 128 are four waves."""
import os
import re
import shutil
import subprocess

import pytest

from axon_amd.kernels import build as B


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="no compiler")
@pytest.mark.parametrize("source, kernel, most", [("attention_mfma.hip", "attention_combine_kernel", 128)])
def test_registers_leave_room_for_the_waves(tmp_path, source, kernel, most):
    out = tmp_path / "device.s"
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    done = subprocess.run([hipcc, *B.HIP_FLAGS, B.DTYPE_FLAG["bfloat16"], "-I", B.CSRC, "-S", "--cuda-device-only", "-o", str(out),
                           os.path.join(B.CSRC, source)], capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    seen = 0
    for note in re.findall(r"- \.agpr_count:.*?\.wavefront_size:", out.read_text(), re.S):
        field = {k: v for k, v in re.findall(r"\.(\w+):\s+(\S+)", note)}
        if kernel in field["symbol"]:
            seen += 1
            assert int(field["vgpr_count"]) <= most and int(field["private_segment_fixed_size"]) == 0, field
    assert seen
