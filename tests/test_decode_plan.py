"""The decode launch's plan (csrc/decode_plan.h, host code without HIP),
compiled here and run on the CPU: tests/native/decode_plan_check.cpp walks
shapes, split hints and workspace sizes."""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "paged_tierkv_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_plans_fit_and_deterministic_plans_follow_the_shape(tmp_path):
    exe = tmp_path / "decode_plan_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "native", "decode_plan_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
    assert " bad 0" in res.stdout and "(two plans 0)" not in res.stdout
