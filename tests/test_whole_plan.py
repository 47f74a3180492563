"""The plan that deals row groups of 128 rows whole, checked over random calls on the CPU, and the rules that choose it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_whole_row_groups_and_runs_cover_every_row_group_once(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = tmp_path / "whole_plan_check"
    csrc = os.path.join(ROOT, "inference_lib_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    os.path.join(ROOT, "tests", "host_fuzz", "whole_plan_check.cpp"), os.path.join(csrc, "hogwild_plan.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
