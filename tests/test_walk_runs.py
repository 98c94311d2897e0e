"""CPU test of the walks' runs of equal cost (gem_amd/csrc/host/walk_runs.h)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_runs_cover_their_pieces_and_number_in_32_bits(tmp_path):
    exe = str(tmp_path / "walk_runs")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "gem_amd", "csrc", "host"),
                    os.path.join(ROOT, "tests", "native", "walk_runs.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout[-2000:]
