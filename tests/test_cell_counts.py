"""A cell's triangles by its vertex count, on the host, for counts from -2^31
to 2^31 - 1 (tests/native/count_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pixel-art-remaster-gpu_amd", "csrc")


def test_triangles_of_any_count(tmp_path):
    exe = tmp_path / "count_check"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O2", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "native", "count_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
