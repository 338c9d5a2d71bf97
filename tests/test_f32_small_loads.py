"""The small f32 kernel counts its loads in flight one by one.  A flat load shares the counter of LDS and makes the compiler
wait for all of them at each use: the kernel's addresses must stay global ones in what the compiler makes of them."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "graph-compiler_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc here")
def test_no_flat_loads(tmp_path):
    out = tmp_path / "gemm_f32.s"
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-O3",
                           "-std=c++17", "-fPIC", "-w", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-S", "--cuda-device-only",
                           os.path.join(CSRC, "kernels", "gemm_f32.hip"), "-o", str(out)])
    bodies = re.findall(r"^(\w*gemm_f32_small_kernel\w*):(.*?)s_endpgm", out.read_text(), re.M | re.S)
    assert len(bodies) == 8  # two layouts of A, two of B, strides within 32 bits and beyond
    for name, body in bodies:
        assert "global_load" in body and "flat_load" not in body, name
