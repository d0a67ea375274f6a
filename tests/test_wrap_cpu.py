"""Wrapping, z-bins, lattice images and grid points of any position (csrc/atm_wrap.h), on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_positions_of_any_size(tmp_path):
    exe = str(tmp_path / "TestWrap")
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17",
                    "-I" + os.path.join(ROOT, "openmm-atmmetaforce-plugin_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "TestWrap.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.strip() == "Done"
