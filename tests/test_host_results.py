"""A program's host copies of its results (hindemith_amd/csrc/host_result.h): a refusal of
pinned memory, or too much of it already, leaves pageable copies and no error."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pinned_budget_and_pageable_fallback(tmp_path):
    exe = tmp_path / "results"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", str(exe),
                    os.path.join(HERE, "host_result_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
