"""The FP64 propagator + Dyson chain on matrix cores (blocks of at most 80 states) at the edges of
its tile classes, Taylor degrees and squarings: gamma-COMPUTE FIDs with step lengths from a small
to a large phase, and pulse programs whose rf phase turns from step to step, whose steps differ in
length, and whose blocks fill every class (2 to 70 states).  Against the oracle, 1e-9 relative L2
(the FP64 bar)."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from blochlib_amd.spinsys import SolidSys
from oracle import oracle as O

pytestmark = pytest.mark.gpu
PW = zcw(1154).subset(np.arange(3, 1154, 420))
MAGIC = workloads.MAGIC_DEG


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# few steps per period make X large (squarings), many make it small (low degrees)
@pytest.mark.parametrize("spins,n,wr", [(1, 2, 9000.0), (2, 200, 30000.0),
                                        (3, 5, 4000.0), (4, 64, 12000.0), (5, 3, 9000.0),
                                        (6, 4, 15000.0), (6, 128, 25000.0), (7, 6, 9000.0),
                                        (7, 40, 15000.0), (8, 3, 15000.0), (8, 24, 20000.0)])
def test_gamma_compute(spins, n, wr):
    sy = workloads.small_cluster(spins, 50 + spins)
    rho, det = sy.op("Ix"), sy.op("Ip")
    print(f"[chain64] S={spins} n={n} wr={wr}", flush=True)
    pw = PW if spins < 8 else PW.subset(np.arange(1))
    g, _ = engine.powder_fid(sy, wr, MAGIC, n * wr, 37, pw, rho, det)
    c, _ = O.powder_fid(sy, wr, MAGIC, n * wr, 37, pw, rho, det)
    assert rel(g, c) < 1e-9


@pytest.mark.parametrize("spins,carbon", [(1, False), (2, False), (3, True), (4, False), (4, True),
                                          (5, False), (6, False), (6, True), (7, True)])
def test_pulse_phases_and_lengths(spins, carbon):
    sy = workloads.small_cluster(spins, 60 + spins)
    if carbon:  # one 13C: its Zeeman states stay apart, and it is pulsed in the second half
        sy = SolidSys(["13C"] + ["1H"] * (spins - 1), list(sy.csa), list(sy.dip), [])
        sy.add_j(140.0, 0, 1)
    rng = np.random.default_rng(spins)
    n = 7
    dt = rng.uniform(0.3e-6, 4.0e-6, n)
    rf = [("1H", np.where(np.arange(n) == 3, 0.0, 70000.0), rng.uniform(0, 6.0, n),
           rng.uniform(-500, 500, n))]
    if carbon:
        rf.append(("13C", np.where(np.arange(n) < 4, 0.0, 45000.0), rng.uniform(0, 6.0, n),
                   np.zeros(n)))
    rho, det = sy.op("Iz"), sy.op("Ip_0")
    print(f"[chain64] pulse S={spins} carbon={carbon}", flush=True)
    g = engine.pulse_fid(sy, 11000.0, MAGIC, dt, 21, PW, rho, det, rf=rf)
    c = O.ptop_fid(sy, 11000.0, MAGIC, n, 21, PW, rho, det, rf=rf, step_dt=dt)
    assert rel(g, c) < 1e-9
