"""The cell pass's walk from a cell to its column, CPU only: tests/cell_walk_check.cpp compiles the
kernel's own function for the host and sweeps it over column groups, the map's end among them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_cell_walk(tmp_path):
    exe = str(tmp_path / "cell_walk_check")
    cmd = ["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
           os.path.join(ROOT, "g-vom_amd", "csrc"), "-x", "hip", os.path.join(ROOT, "tests", "cell_walk_check.cpp"),
           "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
