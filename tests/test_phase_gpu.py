"""Phases of the eigenbasis FID at thousands of radians: uncoupled spins whose shifts (quarters of a
Hz) and hence eigenvalues are exact, against exp(i k w l) in extended precision with the same FP64
w = -2 pi / sw.  A point is a product of at most twelve table factors and seven rotations of groups,
each to 4 eps, and sums of equal terms over the states: 64 eps relative to its size at t = 0.  1, 3, 5 and 7
spins: one wave and four, listed and unlisted elements; FIDs of one, of several and of more than eight
groups of 256 points."""
import numpy as np
import pytest

from blochlib_amd import engine
from blochlib_amd.powder import Powder
from blochlib_amd.spinsys import SolidSys

pytestmark = pytest.mark.gpu
SHIFTS = [20000.25, -17333.75, 4021.5, 11999.25, -301.75, 23456.5, -9876.25]


@pytest.mark.parametrize("spins", [1, 3, 5, 7])
@pytest.mark.parametrize("npts", [200, 1000, 5000])
def test_phases(spins, npts):
    sw = 50000.0
    sy = SolidSys(isotopes=["1H"] * spins,
                  csa=[(SHIFTS[i], 0.0, 0.0, i, 0.0, 0.0, 0.0) for i in range(spins)])
    pw = Powder(np.zeros(1), np.zeros(1), np.zeros(1), np.ones(1))
    print(f"[phase] S={spins} npts={npts}", flush=True)
    f, _ = engine.powder_fid(sy, 0.0, 0.0, sw, npts, pw, sy.op("Ix"), sy.op("Ip"))
    w = np.longdouble(-6.283185307179586476925286766559 / sw)
    ph = np.arange(npts, dtype=np.longdouble)[:, None] * (w * np.array(SHIFTS[:spins], np.longdouble))
    want = ((np.cos(ph) + 1j * np.sin(ph)).sum(1) / (2 * spins))
    err = np.abs(f.astype(np.clongdouble) - want).max()
    print(f"[phase] S={spins} npts={npts}: {float(err):.2e}", flush=True)
    assert abs(want[0] - 0.5) < 1e-15 and err < 64 * 2.0 ** -53 * 0.5
