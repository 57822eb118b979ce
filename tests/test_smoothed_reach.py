"""The reach of smoothed cells over all pairs of cell keys, against the sample
grid that their coverage is taken on (tests/native/reach_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pixel-art-remaster-gpu_amd", "csrc")


def test_grid_holds_every_smoothed_vertex(tmp_path):
    exe = tmp_path / "reach_check"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O2", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "native", "reach_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert out.stdout.split() == ["-48", "86", "-42", "106"]
