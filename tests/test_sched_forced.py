"""CPU test of chunks forced past the level budget while levels are measured in
parts (gem_amd/csrc/host/vsched.h)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("forced") / "sched_forced")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "gem_amd", "csrc", "host"),
                    os.path.join(ROOT, "tests", "native", "sched_forced.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("cap", [1, 100000, 5000000, 10**8])
def test_same_chunks_past_the_budget(exe, cap):
    out = subprocess.run([exe, str(cap)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.endswith("ok\n"), out.stdout
