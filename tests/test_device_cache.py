"""The per-device cache behind the grids of the tile kernels
(csrc/device_cache.h), compiled for the host: one value per device, a failed
query not kept, several threads."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_device_cache(tmp_path):
    exe = tmp_path / "device_cache"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(ROOT, "smoothedparticles.jl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "device_cache.cpp"), "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
