"""The way of the workgroups of a launch in whole row groups and runs, checked over random prompt chunks on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_workgroups_open_only_row_groups_that_exist(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = tmp_path / "whole_walk_check"
    csrc = os.path.join(ROOT, "inference_lib_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    os.path.join(ROOT, "tests", "host_fuzz", "whole_walk_check.cpp"), os.path.join(csrc, "hogwild_plan.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


def test_the_deal_is_the_rule_in_less_time(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = tmp_path / "whole_deal_check"
    csrc = os.path.join(ROOT, "inference_lib_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    os.path.join(ROOT, "tests", "host_fuzz", "whole_deal_check.cpp"), os.path.join(csrc, "hogwild_plan.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
