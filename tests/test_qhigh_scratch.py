"""The order-5/6 kernels keep a visit's factors in registers: with the visit record in
scratch memory every term reads it there once per factor, and how that schedules
decides some percent of the kernel's time."""
import os
import re
import shutil
import subprocess

import pytest

from host_checks import CSRC

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_no_scratch_memory(tmp_path):
    out = str(tmp_path / "qhigh.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", out, os.path.join(CSRC, "qhigh.hip")],
                   check=True, capture_output=True)
    sizes = dict(re.findall(r"\.set (\S*k_qhigh\S*)\.private_seg_size, (\d+)", open(out).read()))
    assert len(sizes) == 3 and set(sizes.values()) == {"0"}, sizes
