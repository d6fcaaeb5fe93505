"""The reciprocal quotient (hindemith_amd/csrc/hs_div.h) at every quotient that lies close
to a midpoint of two floats: the cases its argument leaves to enumeration."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_near_midpoint_quotient(tmp_path):
    exe = tmp_path / "hard"
    flags = ["-O2", "-std=c++17", "-ffp-contract=off", "-Wall"]
    if "fma" in open("/proc/cpuinfo").read():
        flags.append("-mfma")
    subprocess.run(["g++", *flags, "-o", str(exe), os.path.join(HERE, "fast_div_hard_cases.cpp")],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
