"""The rules of the device memory that schedules leave behind, against a made-up runtime (tests/cpp/test_idle_blocks.cpp)."""
import os
import subprocess
from types import SimpleNamespace

import pytest
import torch

from conftest import ROOT
from neutronbench_amd import abi


def test_rules_of_the_kept_memory(tmp_path):
    exe = str(tmp_path / "test_idle_blocks")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "neutronbench_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_idle_blocks.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


@pytest.mark.parametrize("make,args,kwargs", [(torch.empty, (3, 4), {"device": "cuda:0"}),
                                              (torch.empty_like, (SimpleNamespace(device="cuda:1"),), {})])
def test_a_tensor_that_does_not_fit_gets_the_idle_memory(monkeypatch, make, args, kwargs):
    """The allocations of the Python layer: one more try, on the same device, after nts_scratch_trim."""
    log = []

    class Device:
        def __init__(self, device):
            self.device = device

        def __enter__(self):
            log.append(self.device)

        def __exit__(self, *error):
            log.append("left")

    def fails(times):
        def made(*a, **k):
            log.append("make")
            if log.count("make") <= times:
                raise torch.OutOfMemoryError("made up")
            return a, k
        return made

    monkeypatch.setattr(torch.cuda, "device", Device)
    monkeypatch.setattr(abi, "status", lambda name: log.append(name))
    device = kwargs.get("device") or args[0].device
    assert abi.allocate(fails(0), *args, **kwargs) == (args, kwargs) and log == ["make"]
    del log[:]
    assert abi.allocate(fails(1), *args, **kwargs) == (args, kwargs)
    assert log == ["make", device, "nts_scratch_trim", "left", "make"]
    del log[:]
    with pytest.raises(torch.OutOfMemoryError):
        abi.allocate(fails(2), *args, **kwargs)
    assert log.count("make") == 2
