"""The one-pass B and Q products of block pairs of at most 16 states (every block size it meets, a
block paired with itself, a complex detection operator, rho of the autocorrelation form, a general
and a prepared one, runs of steps of every length) and the block Jacobi of blocks above 80 states
(the smallest that takes it, and one whose size leaves absent indices).  Against the oracle: FP64
to 1e-9 relative L2, complex64 to 1e-5 (the bars of the parity and precision tests)."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from oracle import oracle as O

pytestmark = pytest.mark.gpu
PW = zcw(1154)
WR = 12000.0
BARS = (("fp64", 1e-9), ("c64", 1e-5))


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def both(sy, n, npts, pw, rho, det):
    c, _ = O.powder_fid(sy, WR, workloads.MAGIC_DEG, n * WR, npts, pw, rho, det)
    for prec, tol in BARS:
        g, _ = engine.powder_fid(sy, WR, workloads.MAGIC_DEG, n * WR, npts, pw, rho, det,
                                 precision=prec)
        assert rel(g, c) < tol, prec


@pytest.mark.parametrize("ops", ["sym", "general", "complex", "same"])
@pytest.mark.parametrize("spins,K,n", [(1, 2, 8), (2, 1, 33), (3, 40, 64), (4, 5, 17), (5, 3, 16),
                                       (6, 2, 20), (2, 1154, 40)])
def test_small_pairs(spins, K, n, ops):
    sy = workloads.small_cluster(spins, 20 + spins)
    rho = sy.op("Ix" if ops in ("sym", "complex") else "Iy_0+0.5*Iz_0")
    det = sy.op("Ip")
    if ops == "complex":
        det = np.exp(0.7j) * det + 0.2j * sy.op("Iz_0")
    elif ops == "same":  # pairs (I, I) only
        rho, det = sy.op("Iz_0"), sy.op("Iz_0")
    print(f"[pairs] S={spins} K={K} n={n} {ops}", flush=True)
    both(sy, n, 50, PW.subset(np.arange(K) * 7 % 1154), rho, det)


# 9 spins: blocks of 84 and 126 states
@pytest.mark.parametrize("spins,n,K", [(9, 3, 1), (9, 4, 3)])
def test_block_jacobi(spins, n, K):
    sy = workloads.small_cluster(spins, 80 + spins)
    print(f"[block jacobi] S={spins} K={K}", flush=True)
    both(sy, n, 20, PW.subset(np.arange(K) * 101), sy.op("Ix"), sy.op("Ip"))
