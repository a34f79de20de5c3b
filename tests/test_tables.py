"""CPU check of the plan's Hamiltonian tables (quadratic forms of the field direction, one per basis
state and flip-flop pair): rounded once from the exact sums over the interactions."""
import os
import subprocess

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


def test_quadratic_forms_are_rounded_once(tmp_path):
    obj, exe = str(tmp_path / "launch.o"), str(tmp_path / "tables_check")
    subprocess.run(["gcc", "-c", os.path.join(CPP, "fake_launch.c"), "-o", obj], check=True)
    subprocess.run(["g++", "-std=gnu++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(CPP, "tables_check.cpp"), obj, "-o", exe,
                    "-lquadmath", "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("OK"), r.stdout
