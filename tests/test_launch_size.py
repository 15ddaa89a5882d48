"""Block counts of launches that grow with their arguments (tests/cpp/test_launch_size.cpp)."""
import os
import subprocess

from conftest import ROOT


def test_no_launch_of_two_to_the_32_threads(tmp_path):
    exe = str(tmp_path / "test_launch_size")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "neutronbench_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_launch_size.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
