"""A server's cached plan serves a later request of the same system over a much larger powder: the
FID is the solo run's, whichever came first."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from blochlib_amd.serve import FIDServer, Request

pytestmark = pytest.mark.gpu
WR = 12000.0


def test_small_powder_then_large():
    sy = workloads.small_cluster(6, 46)
    pows = [zcw(1154).subset(np.arange(5)), zcw(1154), zcw(1154).subset(np.arange(300))]
    srv = FIDServer()
    try:
        for i, pw in enumerate(pows):
            print(f"[serve] K={len(pw)}", flush=True)
            r = Request(i, sy, WR, workloads.MAGIC_DEG, 64 * WR, 256, pw, sy.op("Ix"), sy.op("Ip"))
            done = srv.run([r])
            assert done[0].error is None
            want, _ = engine.powder_fid(sy, WR, workloads.MAGIC_DEG, 64 * WR, 256, pw, sy.op("Ix"),
                                        sy.op("Ip"))
            assert np.array_equal(done[0].fid, want)
    finally:
        srv.close()
