"""The slice loop's element-wise and k-space kernels keep what they compute in
registers: none of them is compiled with scratch memory."""
import os
import re
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "quickpic-opensource_amd")
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_slice_kernels_use_no_scratch(tmp_path):
    out = str(tmp_path / "fused.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
                    "-munsafe-fp-atomics", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-w", "--offload-device-only", "-S",
                    os.path.join(PKG, "csrc", "qp_fused.hip"), "-o", out], check=True)
    asm = open(out).read()
    sizes = dict(re.findall(r"\.amdhsa_kernel (\S+).*?private_segment_fixed_size (\d+)", asm, re.S))
    assert len(sizes) >= 8
    assert {k: v for k, v in sizes.items() if v != "0"} == {}
