"""Where the lanes of one wave hand values to one another through LDS without
a workgroup barrier, the order of the stores and the loads must be visible to
the compiler: s_waitcnt and wave_barrier are no memory operations to it, and
the two sides may have access types that do not alias.  The kernels' LLVM IR
must therefore hold a release fence before and an acquire fence after each
wave barrier.  Compiles two sources for the device, no GPU."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("source,kernel", [("quant.hip", "quantize_q8_0_kernel"), ("strip16.hip", "strip16_kernel")])
def test_wave_handoffs_are_fenced(tmp_path, source, kernel):
    csrc = os.path.join(ROOT, "sam.cpp_amd", "csrc")
    out = tmp_path / "kernels.ll"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-emit-llvm", "-S",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"),
                    "-I" + csrc, "-x", "hip", "-o", str(out), os.path.join(csrc, source)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL, timeout=300)
    bodies = re.findall(r"^define [^\n]*" + kernel + r"[^\n]*\{\n(.*?)^\}", out.read_text(), re.M | re.S)
    assert bodies
    for body in bodies:
        marks = re.findall(r'call void @llvm\.amdgcn\.wave\.barrier|fence syncscope\("wavefront"\) (?:release|acquire)', body)
        barriers = [i for i, m in enumerate(marks) if "barrier" in m]
        assert barriers
        for i in barriers:
            assert i > 0 and marks[i - 1].endswith("release") and marks[i + 1:] and marks[i + 1].endswith("acquire")
