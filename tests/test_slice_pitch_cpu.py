"""CPU check of the row pitch of the K slices' sums (kudnn_slice_pitch in kudnn_amd/csrc/kernels.h): wider rows of sums never
make the allocation-free entry point refuse a call that narrower ones let through (tests/cpp/test_slice_pitch.cpp)."""
import os
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_slice_pitch_refuses_nothing(tmp_path):
    exe = tmp_path / "test_slice_pitch"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", str(ROOT / "kudnn_amd" / "csrc"),
                    "-I", str(ROOT / "include"), "-I", rocm + "/include",
                    str(ROOT / "tests" / "cpp" / "test_slice_pitch.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
