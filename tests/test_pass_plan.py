"""The sizes of a pass's launches (forkerrenderer_amd/csrc/pass_plan.hpp):
tests/pass_plan_check.cpp, built with the host compiler."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "forkerrenderer_amd", "csrc")


def test_pass_plan(tmp_path):
    exe = str(tmp_path / "pass_plan_check")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, os.path.join(HERE, "pass_plan_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    if r.returncode != 0:
        pytest.fail("build failed:\n" + r.stdout + r.stderr)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
