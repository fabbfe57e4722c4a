"""The threshold rounds' decision of picks (fpsample_amd/csrc/fps_rounds_bound.hpp).

tests/rounds_check.cpp restates the rounds on the host with the bounds and steps that the
kernels take, and compares every pick with the loop that takes one pick per pass, on clouds small
enough that one round can hold every point: wide scales, duplicates, special values, both tie
rules, runs in parts.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_rounds_take_the_picks_of_the_plain_loop(tmp_path):
    exe = tmp_path / "rounds_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "fpsample_amd", "csrc"),
                    os.path.join(ROOT, "tests", "rounds_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout + out.stderr
