"""The predictor of the range-gated FP64 kernels against the reference's order of
operations, bit for bit (zeros' signs included), on the CPU: the device functions
compiled as plain C++ (tests/host/check_predictor.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_scaled_predictor_has_the_same_bits(tmp_path):
    if not shutil.which("g++") or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no g++ or HIP headers")
    exe = str(tmp_path / "check")
    # (no multiply-adds but those in the source)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-w",
                    "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"), "-o", exe,
                    os.path.join(ROOT, "tests", "host", "check_predictor.cpp"), "-lm"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stdout
