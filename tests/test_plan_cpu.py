"""How transfers are cut into launches and how many workgroups they take.

Builds tests/native/plan_check.cpp with g++ against flexkv_amd/csrc/kv_plan.h
(header-only, no HIP) and runs it.  No device is involved.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_plans(tmp_path):
    exe = tmp_path / "plan_check"
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "flexkv_amd", "csrc"),
           os.path.join(ROOT, "tests", "native", "plan_check.cpp"), "-o", str(exe)]
    build = subprocess.run(cmd, capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and "FAIL" not in res.stdout, res.stdout + res.stderr
    assert res.stdout.count("ok:") == 20
