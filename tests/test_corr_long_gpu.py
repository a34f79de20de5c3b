"""FIDs too long to be held on chip, on both sides of the length where a crystallite's partial sums
reach their limit and the correlation's segments grow, with a segment count that does not divide.
Against the oracle: a period phase of 20 states is exact to about 20 eps = 4e-15, times 2200 periods
on either side, so 1e-10 relative L2."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from oracle import oracle as O

pytestmark = pytest.mark.gpu
WR = 12000.0


@pytest.mark.parametrize("n,npts", [(32, 60000), (32, 70000), (45, 70001)])
def test_long_fid(n, npts):
    sy = workloads.small_cluster(6, 30)
    pw = zcw(1154).subset(np.array([100, 801]))
    rho, det = sy.op("Ix"), sy.op("Ip")
    print(f"[corr] n={n} npts={npts}", flush=True)
    c, _ = O.powder_fid(sy, WR, workloads.MAGIC_DEG, n * WR, npts, pw, rho, det)
    g, _ = engine.powder_fid(sy, WR, workloads.MAGIC_DEG, n * WR, npts, pw, rho, det)
    assert np.linalg.norm(g - c) < 1e-10 * np.linalg.norm(c)


# step counts whose periods are only just held on chip, one element at a time
@pytest.mark.parametrize("n,npts", [(513, 700), (1024, 2100), (1025, 1500), (2047, 2500), (2048, 900)])
def test_many_steps(n, npts):
    sy = workloads.small_cluster(3, 33)
    pw = zcw(1154).subset(np.array([100, 801]))
    rho, det = sy.op("Iy_0+0.5*Iz_1"), sy.op("Ip")
    print(f"[corr] n={n} npts={npts}", flush=True)
    c, _ = O.powder_fid(sy, 100.0, workloads.MAGIC_DEG, n * 100.0, npts, pw, rho, det)
    g, _ = engine.powder_fid(sy, 100.0, workloads.MAGIC_DEG, n * 100.0, npts, pw, rho, det)
    assert np.linalg.norm(g - c) < 1e-10 * np.linalg.norm(c)
