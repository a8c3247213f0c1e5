"""Host check of the correctly rounded trigonometry (voxelyze_amd/csrc/vx_math.h) against binary128:
tests/cpp/cr_trig.cpp, compiled with g++ (no GPU needed)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_trig_is_correctly_rounded(tmp_path):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("g++ or the HIP headers not available")
    exe = tmp_path / "cr_trig"
    src = os.path.join(ROOT, "tests", "cpp", "cr_trig.cpp")
    r = subprocess.run(["g++", "-O2", "-std=gnu++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I",
                        "/opt/rocm/include", src, "-o", str(exe), "-lquadmath"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=110)
    print(r.stdout[-2000:])
    assert r.returncode == 0 and r.stdout.strip().endswith("\n0 failures"), r.stdout[-2000:]
