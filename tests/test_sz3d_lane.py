"""Host replay of the lane kernels' work split: the 3-D codec with block side 4,
and the carries of the 1-D index (tests/sz3d_lane_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lane_work_split(tmp_path):
    exe = str(tmp_path / "sz3d_lane_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "zccl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "sz3d_lane_check.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok ")
