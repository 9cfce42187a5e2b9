"""The library's host code against HIP calls that fail or wait, on the CPU: its
sources are compiled for the host alone and linked with a stand-in for the HIP runtime
(tests/host/hip_on_host.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def run_check(tmp_path, check, library, *args):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    src = [os.path.join(ROOT, "tests", "host", f) for f in ("hip_on_host.cpp", check)]
    src.append(os.path.join(ROOT, "hydro_amd", "csrc", library))
    objs = []
    for s in src:
        objs.append(str(tmp_path / (os.path.basename(s) + ".o")))
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-fPIC", "-std=c++17",
                        "-Wno-unused-result", "-c", s, "-o", objs[-1]], check=True)
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-o", exe, *objs, "-lpthread", "-lm"], check=True)
    out = subprocess.run([exe, *args], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
    return out.stdout


def test_batch_autotune_puts_the_controls_back(tmp_path):
    run_check(tmp_path, "check_batch_autotune.cpp", "hydro_batch.cpp")


@pytest.mark.parametrize("check", ["no_pinned_memory", "devices", "busy_upload", "busy_download"])
def test_staged_copies(tmp_path, check):
    run_check(tmp_path, "check_stage.cpp", "hydro_stage.cpp", check)


def test_batch_grows_with_another_device_current(tmp_path):
    run_check(tmp_path, "check_batch_devices.cpp", "hydro_batch.cpp")
