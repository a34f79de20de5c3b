"""CPU checks of the device memory the host code takes, keeps and gives back: the engine's host
code (blochlib_amd/csrc/blfid_host.cpp) on a runtime without a device, whose allocations are a
table and whose kernels do nothing (tests/cpp/fake_hip.h)."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
CHECKS = ["workspace", "release", "reset", "budget", "age", "host_memory", "accepted", "copies", "footprint", "steps"]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("memory")
    obj, out = str(d / "launch.o"), str(d / "memory_check")
    subprocess.run(["gcc", "-c", os.path.join(CPP, "fake_launch.c"), "-o", obj], check=True)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(CPP, "memory_check.cpp"), obj,
                    "-o", out, "-lpthread"], check=True)
    return out


@pytest.mark.parametrize("check", CHECKS)
def test_memory(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("OK"), r.stdout
