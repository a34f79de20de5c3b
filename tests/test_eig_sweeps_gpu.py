"""Blocks above 80 states whose Jacobi sweeps do not end within those launched over the whole device
are finished by one workgroup each: gamma-COMPUTE (FP64 and complex64), static and pulse-program
FIDs of a few launched sweeps against the oracle, to the bars of the large-block tests, and against
the default number of sweeps (the same rotations: to the rounding of the solver, 256 eps = 6e-14 a
sweep, ten sweeps)."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from oracle import oracle as O

pytestmark = pytest.mark.gpu
WR, MAGIC = 12000.0, workloads.MAGIC_DEG
PW = zcw(1154).subset(np.array([5, 700]))


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def runs(p, pw, rho, det, want, tol):
    try:
        p.set_operators(rho, det)
        p.set_powder(pw)
        ref = None
        for sweeps in (0, 1, 3, 5):
            print(f"[sweeps] {sweeps}", flush=True)
            p.set_eig_sweeps(sweeps)
            p.run()
            f = p.fetch()
            assert rel(f, want) < tol, sweeps
            ref = f if ref is None else ref
            assert rel(f, ref) < (1e-12 if tol < 1e-8 else 1e-6), sweeps
        with pytest.raises(engine.EngineError):
            p.set_eig_sweeps(13)
    finally:
        p.close()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("c64", 1e-5)])
def test_gamma_compute(precision, tol):
    sy = workloads.small_cluster(9, 89)
    rho, det, n = sy.op("Ix"), sy.op("Ip"), 3
    pw = PW.subset(np.array([0]))
    want, _ = O.powder_fid(sy, WR, MAGIC, n * WR, 20, pw, rho, det)
    runs(engine.Plan(sy, WR, MAGIC, n * WR, 20, precision=precision), pw, rho, det, want, tol)


def test_pulse_program():
    sy = workloads.small_cluster(7, 87)
    rf = [("1H", np.full(3, 90000.0), np.array([0.1, 0.9, 0.4]), np.full(3, 500.0))]
    rho, det = sy.op("Ix"), sy.op("Ip")
    want = O.ptop_fid(sy, 30000.0, MAGIC, 3, 20, PW, rho, det, rf=rf)
    runs(engine.Plan.ptop(sy, 30000.0, MAGIC, 3, 20, rf), PW, rho, det, want, 1e-11)


def test_static():
    sy = workloads.small_cluster(9, 89)
    rho, det = sy.op("Ix"), sy.op("Ip")
    pw = PW.subset(np.array([0]))
    want, _ = O.powder_fid(sy, 0.0, 0.0, 50000.0, 20, pw, rho, det)
    runs(engine.Plan(sy, 0.0, 0.0, 50000.0, 20), pw, rho, det, want, 1e-11)
