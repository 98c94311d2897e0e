"""CPU test of the numbers that set-aside rows and their pieces get
(gem_amd/csrc/host/heavy_pieces.h), past both tables' ends and past 2^32."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("heavy") / "heavy_pieces")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "gem_amd", "csrc", "host"),
                    os.path.join(ROOT, "tests", "native", "heavy_pieces.cpp"), "-o", exe], check=True)
    return exe


def test_every_piece_numbered_once(exe):
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout


def test_check_finds_numbers_in_32_bits(exe):
    out = subprocess.run([exe, "control"], capture_output=True, text=True, timeout=120)
    assert out.returncode > 0, out.stdout
