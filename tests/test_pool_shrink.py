"""CPU test of the caching allocator's in-place shrink (gem_amd/csrc/host/pool_core.h)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_shrink(tmp_path):
    exe = str(tmp_path / "pool_shrink")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "gem_amd", "csrc", "host"),
                    os.path.join(ROOT, "tests", "native", "pool_shrink.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
