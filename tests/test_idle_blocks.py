"""The rules of the device memory that schedules leave behind, against a made-up runtime (tests/cpp/test_idle_blocks.cpp)."""
import os
import subprocess

from conftest import ROOT


def test_rules_of_the_kept_memory(tmp_path):
    exe = str(tmp_path / "test_idle_blocks")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "neutronbench_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_idle_blocks.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
