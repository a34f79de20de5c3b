"""The eigenbasis FID (k_static_fid) at the edges of its point groups, element list and tile
classes, against the oracle: groups of 256 points held four or eight at a time (a second batch
from 2049 points on), the squeezed element list of small packed blocks, phase tables in LDS and
in the scratch slot.  Tolerance 1e-9 relative L2, the FP64 bar of the static and pulse paths."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from oracle import oracle as O

pytestmark = pytest.mark.gpu
PW = zcw(1154).subset(np.arange(5, 1154, 400))


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("spins,npts", [(1, 1), (2, 255), (3, 256), (3, 2049), (4, 257),
                                        (5, 1024), (6, 1025), (7, 300), (8, 513), (9, 40)])
def test_static(spins, npts):
    sy = workloads.small_cluster(spins, 70 + spins)
    rho, det = sy.op("Ix"), sy.op("Ip")
    print(f"[eigfid] static S={spins} npts={npts}", flush=True)
    g, _ = engine.powder_fid(sy, 0.0, 0.0, 60000.0, npts, PW, rho, det)
    c, _ = O.powder_fid(sy, 0.0, 0.0, 60000.0, npts, PW, rho, det)
    assert rel(g, c) < 1e-9


@pytest.mark.parametrize("spins,npts", [(2, 2300), (4, 511), (5, 1030), (6, 260)])
def test_pulse_program(spins, npts):
    sy = workloads.small_cluster(spins, 90 + spins)
    rho, det = sy.op("Iz"), sy.op("Ip_0")
    rf = workloads.phase_alternating_rf("1H", 16, 60000.0, 2)
    print(f"[eigfid] pulse S={spins} npts={npts}", flush=True)
    g = engine.ptop_fid(sy, 10000.0, workloads.MAGIC_DEG, 16, npts, PW, rho, det, rf=rf)
    c = O.ptop_fid(sy, 10000.0, workloads.MAGIC_DEG, 16, npts, PW, rho, det, rf=rf)
    assert rel(g, c) < 1e-9
