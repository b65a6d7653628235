"""The thread order of the whole-grid passes in the forms that the adjoint and the fused
engine use, and for blocks past a stripe's rows, checked on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_fronts_phases_and_idle_blocks(tmp_path):
    exe = str(tmp_path / "row_cover_edges")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "row_cover_edges.cpp"), "-o", exe], check=True,
                   capture_output=True, timeout=600)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "row cover edges ok" in out.stdout, out.stdout + out.stderr
