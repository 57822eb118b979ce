"""The graph kernel's strips and its and the raster's 4-byte pixel loads, on
the host: no load that begins inside an item ends past it
(tests/native/strip_check.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pixel-art-remaster-gpu_amd", "csrc")


@pytest.mark.timeout(300)
def test_pixel_loads_stay_inside_their_item(tmp_path):
    exe = tmp_path / "strip_check"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O2", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "native", "strip_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    loads, left_out = map(int, out.stdout.split())
    assert loads > 1_000_000 and left_out > 10_000


def test_reserved_strips_cover_every_batch(tmp_path):
    exe = tmp_path / "reserve_check"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O2", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "native", "reserve_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    batches, most = map(int, out.stdout.split())
    assert batches == 60000 and most > 500
