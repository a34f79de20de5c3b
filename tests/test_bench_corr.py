"""bench.py's flop count of the correlation kernel is the engine's own at every step count."""
import os
import subprocess

import bench

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


def test_counts_as_the_engine(tmp_path):
    obj, exe = str(tmp_path / "launch.o"), str(tmp_path / "corr_flops")
    subprocess.run(["gcc", "-c", os.path.join(CPP, "fake_launch.c"), "-o", obj], check=True)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(CPP, "corr_flops.cpp"), obj, "-o", exe,
                    "-lpthread"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True).stdout
    rows = [ln.split() for ln in out.splitlines()]
    assert len(rows) == 600
    for n, ln, general, auto in rows:
        n, length = int(n), (1 << int(ln)) if int(ln) else 0
        assert bench.corr_transform_length(n) == length, n
        assert bench.corr_flops_per_elem(n, 1000, False, length) == float(general), n
        assert bench.corr_flops_per_elem(n, 1000, True, length) == float(auto), n
