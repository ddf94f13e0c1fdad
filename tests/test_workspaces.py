"""Workspaces of the azimuth-ordered cast, the cell pass and the slot clear, CPU only:
tests/workspace_check.cpp compares what the kernels index with what is allocated and calls the
launchers with buffers one word short, which they must refuse before any device work."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "g-vom_amd")


def test_workspaces_and_launcher_refusals(tmp_path):
    assert os.path.exists(os.path.join(PKG, "libgvom_hip.so")), "build the library first (__graft_entry__.build())"
    exe = str(tmp_path / "workspace_check")
    cmd = ["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I", os.path.join(PKG, "csrc"),
           os.path.join(ROOT, "tests", "workspace_check.cpp"), "-L", PKG, "-lgvom_hip", f"-Wl,-rpath,{PKG}", "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
