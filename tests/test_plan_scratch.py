"""The rules of a schedule's scratch, on a made-up device (tests/cpp/test_plan_scratch.cpp)."""
import os
import subprocess

from conftest import ROOT


def test_rules_of_a_schedules_scratch(tmp_path):
    exe = str(tmp_path / "test_plan_scratch")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "neutronbench_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_plan_scratch.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
