"""The FP64 forms of the one- and few-tile kernels against the oracle at a tight bar: fused chains of
every tile class up to 64 states (gamma-COMPUTE and rf), correlations at padded, unpadded and direct
step counts, autocorrelation and general rho, static and pulse-program FIDs.

A step's propagator and product round to about b eps of a b-state block (64 eps = 7e-15 at most), a
period is at most 64 steps in a row and a FID at most 64 periods, whose phase errors add up:
64 (sqrt(64) 7e-15) = 3.6e-12, on either side: 1e-11 relative L2."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from oracle import oracle as O

pytestmark = pytest.mark.gpu
MAGIC = workloads.MAGIC_DEG
TOL = 1e-11


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("spins,n,npts", [(2, 64, 500), (3, 8, 400), (4, 9, 500), (4, 16, 500),
                                          (4, 45, 600), (5, 33, 300), (6, 17, 300), (6, 32, 500),
                                          (7, 12, 200), (8, 10, 100)])
def test_gamma_compute(spins, n, npts, general):
    sy = workloads.small_cluster(spins, 60 + spins)
    rho, det = sy.op("Iy_0+0.5*Iz_1" if general else "Ix"), sy.op("Ip")
    pw = zcw(1154).subset(np.arange(3) * 301 + n)
    c, _ = O.powder_fid(sy, 12000.0, MAGIC, n * 12000.0, npts, pw, rho, det)
    g, _ = engine.powder_fid(sy, 12000.0, MAGIC, n * 12000.0, npts, pw, rho, det)
    print(f"[bars] S={spins} n={n} {rel(g, c):.2e}", flush=True)
    assert rel(g, c) < TOL


@pytest.mark.parametrize("spins", [2, 3, 4, 5, 6])
def test_pulse_program(spins):
    sy = workloads.small_cluster(spins, 70 + spins)
    n = 16
    rf = [("1H", np.full(n, 80000.0), np.repeat([0.0, 0.6, 1.9, 0.6], 4), np.full(n, 300.0))]
    pw = zcw(1154).subset(np.arange(3) * 301)
    c = O.ptop_fid(sy, 20000.0, MAGIC, n, 64, pw, sy.op("Ix"), sy.op("Ip"), rf=rf)
    g = engine.ptop_fid(sy, 20000.0, MAGIC, n, 64, pw, sy.op("Ix"), sy.op("Ip"), rf=rf)
    print(f"[bars] rf S={spins} {rel(g, c):.2e}", flush=True)
    assert rel(g, c) < TOL


@pytest.mark.parametrize("spins,npts", [(2, 600), (4, 1500), (6, 300)])
def test_static(spins, npts):
    sy = workloads.small_cluster(spins, 75 + spins)
    pw = zcw(1154).subset(np.arange(5) * 201)
    c, _ = O.powder_fid(sy, 0.0, 0.0, 50000.0, npts, pw, sy.op("Ix"), sy.op("Ip"))
    g, _ = engine.powder_fid(sy, 0.0, 0.0, 50000.0, npts, pw, sy.op("Ix"), sy.op("Ip"))
    print(f"[bars] static S={spins} {rel(g, c):.2e}", flush=True)
    assert rel(g, c) < TOL
