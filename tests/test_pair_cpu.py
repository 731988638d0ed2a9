"""A face's flux from both of its cells (zfv_pair.hpp) against two evaluations, on
the CPU: the device header compiles as plain C++ with the qualifier stand-ins of
tests/hostshim (tests/pair_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_flux_pair_is_both_evaluations_and_made_once(tmp_path):
    exe = tmp_path / "pair_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "tests", "hostshim"),
                    "-I", os.path.join(ROOT, "zephyr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "pair_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
