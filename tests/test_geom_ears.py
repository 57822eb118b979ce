"""The lane-wise ear clipping, the polygon shapes and the T-junction corners
against the routines they stand for, on the host (tests/native/ear_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pixel-art-remaster-gpu_amd", "csrc")


def test_ears_and_corners(tmp_path):
    exe = tmp_path / "ear_check"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-O2", "-std=c++17", "-I", CSRC,
                    "-x", "hip", os.path.join(HERE, "native", "ear_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    polygons, strict, cells = map(int, out.stdout.split())
    assert polygons == 400000 and strict > 1000 and cells > 5000
