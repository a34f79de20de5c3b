"""The products of larger blocks with a density operator of their own, and pulse programs on blocks
above 80 states, against the oracle.

A general rho and a complex detection operator (R formed beside Q, sparse rows of rho) and a
prepared or state rho (dense blocks per crystallite) on pairs of every tile class above 16 states:
7 spins (blocks of 21 and 35), 8 (28, 56, 70) and 9 (36, 84, 126).  Pulse programs of seven protons
(one block of 128 states) and eight (256, the largest): rf whose phase changes or not, even and odd
step counts (the running product alternates between two slots), FIDs, states and their traces.

A product of blocks of up to 256 states rounds to at most 256 eps = 6e-14 of its norm, and a FID
takes some fifty of them one after the other: FP64 to 1e-11 relative L2; complex64 to 1e-5, the bar
of the precision tests."""
import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw
from oracle import oracle as O

pytestmark = pytest.mark.gpu
WR, MAGIC = 12000.0, workloads.MAGIC_DEG
BARS = (("fp64", 1e-11), ("c64", 1e-5))


def rel(a, b):
    return np.linalg.norm(np.ravel(a - b)) / max(np.linalg.norm(np.ravel(b)), 1e-300)


def case(spins, K):
    sy = workloads.small_cluster(spins, 80 + spins)
    rho = sy.op("Iy_0+0.5*Iz_1")
    det = np.exp(0.7j) * sy.op("Ip") + 0.2j * sy.op("Iz_0")
    return sy, rho, det, zcw(1154).subset(np.arange(K) * 101)


@pytest.mark.parametrize("spins,n,K", [(7, 6, 3), (8, 4, 2), (9, 3, 1)])
def test_general_rho(spins, n, K):
    sy, rho, det, pw = case(spins, K)
    c, _ = O.powder_fid(sy, WR, MAGIC, n * WR, 20, pw, rho, det)
    for prec, tol in BARS:
        print(f"[large] general rho S={spins} {prec}", flush=True)
        g, _ = engine.powder_fid(sy, WR, MAGIC, n * WR, 20, pw, rho, det, precision=prec)
        assert rel(g, c) < tol, prec


# delays only: the preparation keeps the magnetisation blocks (up to 126 states)
@pytest.mark.parametrize("spins,n,K", [(6, 8, 3), (7, 6, 3), (8, 4, 2), (9, 3, 1)])
def test_prepared_rho(spins, n, K):
    sy, rho, det, pw = case(spins, K)
    dts = np.array([1.0e-6, 2.5e-6, 0.5e-6])
    c, _ = O.prep_fid(sy, WR, MAGIC, n * WR, 20, pw, rho, det, dts, t0=float(dts.sum()))
    for prec, tol in BARS:
        print(f"[large] prepared rho S={spins} {prec}", flush=True)
        g, _ = engine.prep_fid(sy, WR, MAGIC, n * WR, 20, pw, rho, det, dts, precision=prec)
        assert rel(g, c) < tol, prec


def rf_of(n, phase):
    return [("1H", np.full(n, 90000.0), np.linspace(0.2, 2.0, n) if phase else np.full(n, 0.3),
             np.full(n, 500.0))]


# seven protons under a pulse: one block of 128 states, then their rho in blocks of up to 35
@pytest.mark.parametrize("phase", [False, True])
@pytest.mark.parametrize("nsteps", [1, 4, 5])
def test_pulses_then_fid(nsteps, phase):
    sy, _, det, pw = case(7, 2)
    dts, rf = np.full(nsteps, 0.8e-6), rf_of(nsteps, phase)
    c, _ = O.prep_fid(sy, WR, MAGIC, 6 * WR, 20, pw, sy.op("Iz"), det, dts, rf=rf,
                      t0=float(dts.sum()))
    for prec, tol in BARS:
        print(f"[large] pulses then FID steps={nsteps} phase={phase} {prec}", flush=True)
        g, _ = engine.prep_fid(sy, WR, MAGIC, 6 * WR, 20, pw, sy.op("Iz"), det, dts, rf=rf,
                               precision=prec)
        assert rel(g, c) < tol, prec


@pytest.mark.parametrize("phase", [False, True])
@pytest.mark.parametrize("spins,n,K", [(7, 4, 2), (7, 5, 3), (8, 3, 1), (8, 2, 1)])
def test_pulse_program_fid(spins, n, K, phase):
    sy, _, det, pw = case(spins, K)
    rf = rf_of(n, phase)
    print(f"[large] pulse program S={spins} n={n} phase={phase}", flush=True)
    c = O.ptop_fid(sy, 30000.0, MAGIC, n, 20, pw, sy.op("Ix"), det, rf=rf)
    g = engine.ptop_fid(sy, 30000.0, MAGIC, n, 20, pw, sy.op("Ix"), det, rf=rf)
    assert rel(g, c) < 1e-11


@pytest.mark.parametrize("nsteps,repeat", [(4, 1), (5, 3)])
def test_state_through_pulses(nsteps, repeat):
    sy, rho, det, pw = case(7, 2)
    dts, rf = np.array([0.8e-6, 1.1e-6, 0.4e-6, 0.9e-6, 0.7e-6])[:nsteps], rf_of(nsteps, True)
    print(f"[large] state steps={nsteps} repeat={repeat}", flush=True)
    st = engine.State(sy.spins, pw)
    try:
        st.set(rho)
        st.apply(sy, WR, MAGIC, dts, rf=rf, repeat=repeat)
        got, tr = st.fetch(), st.trace(det)
        want = O.state_apply(sy, WR, MAGIC, dts, pw, np.broadcast_to(rho, got.shape).copy(), rf=rf,
                             repeat=repeat)
        assert rel(got, want) < 1e-11
        t = sum(w * np.trace(r @ det) for w, r in zip(pw.weight, want)) / np.trace(det @ det.conj().T)
        assert abs(tr - t) < 1e-11 * max(abs(t), 1.0)
        c, _ = O.state_fid(sy, WR, MAGIC, 6 * WR, 20, pw, want, det)
        for prec, tol in BARS:
            g, _ = engine.state_fid(sy, WR, MAGIC, 6 * WR, 20, pw, st, det, precision=prec)
            assert rel(g, c) < tol, prec
    finally:
        st.close()
