"""The correlation at step counts that are no power of two: zero-padded transforms from 9 to 256
steps per period (the edges of every transform length), the direct sum outside, with tables of
period phases that fit at once and in parts, FIDs held in registers and longer ones; rho of the
autocorrelation form and a general one.  Against the oracle: FP64 to 1e-9 relative L2, complex64
to 1e-5 (the bars of the parity and precision tests)."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from oracle import oracle as O

pytestmark = pytest.mark.gpu
PW = zcw(1154).subset(np.arange(11, 1154, 300))
WR = 12000.0


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("n,npts", [(8, 100), (9, 300), (15, 1024), (17, 40), (31, 257), (33, 2048),
                                    (45, 777), (63, 64), (65, 1100), (100, 2100), (127, 130),
                                    (129, 500), (200, 1000), (255, 1024), (257, 300),
                                    (16, 1024), (32, 2048)])
def test_steps(n, npts, general):
    sy = workloads.small_cluster(4, 30 + n % 7)
    rho, det = sy.op("Iy_0+Iz_1" if general else "Ix"), sy.op("Ip")
    if general:
        det = det + 0.3 * sy.op("Iz_0")  # elements with a reverse element
    print(f"[corr] n={n} npts={npts} general={general}", flush=True)
    c, _ = O.powder_fid(sy, WR, workloads.MAGIC_DEG, n * WR, npts, PW, rho, det)
    for prec, tol in (("fp64", 1e-9), ("c64", 1e-5)):
        g, _ = engine.powder_fid(sy, WR, workloads.MAGIC_DEG, n * WR, npts, PW, rho, det,
                                 precision=prec)
        assert rel(g, c) < tol, prec
