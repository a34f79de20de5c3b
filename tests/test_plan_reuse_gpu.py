"""Device memory kept between plans: one-call FIDs of alternating sizes, from one thread and from
four threads at once, give the same FID bit for bit whichever block their storage comes from, and
so does a plan whose powder shrinks and grows."""
import threading

import numpy as np
import pytest

from blochlib_amd import engine, workloads
from blochlib_amd.powder import zcw

pytestmark = pytest.mark.gpu
PW = zcw(1154)


def call(spins, K, wr, precision):
    sy = workloads.small_cluster(spins, 40 + spins)
    pw = PW.subset(np.arange(K) * 3 % 1154)
    f, _ = engine.powder_fid(sy, wr, workloads.MAGIC_DEG if wr else 0.0, 32 * 12000.0, 130, pw,
                             sy.op("Ix"), sy.op("Ip"), precision=precision)
    return f


CALLS = [(2, 1, 12000.0, "fp64"), (5, 300, 12000.0, "c64"), (3, 70, 0.0, "fp64"),
         (6, 90, 12000.0, "fp64"), (4, 1154, 0.0, "fp64"), (2, 500, 12000.0, "c64")]


@pytest.mark.parametrize("threads", [1, 4])
def test_calls_in_any_order(threads):
    ref = [call(*c) for c in CALLS]
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for i in rng.permutation(len(CALLS) * 3) % len(CALLS):
            if not np.array_equal(call(*CALLS[i]), ref[i]):
                bad.append((k, CALLS[i]))

    print(f"[reuse] {threads} threads", flush=True)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_powder_of_changing_size():
    sy = workloads.small_cluster(4, 44)
    p = engine.Plan(sy, 12000.0, workloads.MAGIC_DEG, 32 * 12000.0, 100)
    try:
        for K in (3, 700, 1, 1154, 64):
            pw = PW.subset(np.arange(K))
            f = p.powder_fid(pw, sy.op("Ix"), sy.op("Ip"))
            g, _ = engine.powder_fid(sy, 12000.0, workloads.MAGIC_DEG, 32 * 12000.0, 100, pw,
                                     sy.op("Ix"), sy.op("Ip"))
            assert np.array_equal(f, g), K
    finally:
        p.close()
