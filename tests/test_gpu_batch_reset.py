"""A member of a live batch gets a new state through its own handle, and the
batch goes on without a wait in between: its stages come after the member's
upload (which does not wait), its prepared forces and its asynchronous pos
write, whatever call brought the state to the device."""
import numpy as np
import pytest

import bdk
from common import params, positions
from test_gpu_serve import overlapping

pytestmark = pytest.mark.gpu

SIZES = [(12000, 11000, 200.0, 256, 5), (300, 250, 40.0, 64, 6), (2000, 1000, 80.0, 90, 7)]


def make(prec, k, seed=None):
    n1, n2, L, Z, s0 = SIZES[k]
    bp, _ = params(n1=n1, n2=n2, L=L, Z=Z, scheme=bdk.TSC, lam=10.0, precision=prec, seed=s0, max_pair_wca=1e300)
    d = bdk.derived(bp)
    # a lattice: far from overlap, and quick to make
    m = int(np.ceil(np.sqrt(n1 + n2)))
    x = (np.stack(np.meshgrid(np.arange(m), np.arange(m)), -1).reshape(-1, 2)[:n1 + n2] + 0.5) * (L / m)
    x += np.random.default_rng(seed or s0).uniform(-0.05, 0.05, x.shape)
    git = np.clip(np.floor(x / d["B"]), 0, d["nc"] - 1).astype(np.int32)
    return bp, git, x - git * d["B"]


def start(prec, k):
    bp, git, rel = make(prec, k)
    s = bdk.RunDynamik(bp)
    s.set_positions(git, rel)
    return s


@pytest.mark.parametrize("prec", [bdk.FP32, bdk.FP64])
@pytest.mark.parametrize("how", ["prepare", "pos write", "forces", "both"])
@pytest.mark.parametrize("which", [(0,), (1, 2), (0, 1, 2)])
def test_new_state_in_a_live_batch(prec, how, which, tmp_path):
    print("case: new state in a live batch prec=%d by %s, members %s" % (prec, how, which), flush=True)
    members = [start(prec, k) for k in range(3)]
    alone = [start(prec, k) for k in range(3)]
    b = bdk.Batch(members)
    b.run_steps(5)
    b.sync()
    for s in alone:
        s.run_steps(5)
    for rnd in (1, 2):
        for k in which:
            _, git, rel = make(prec, k, 100 * rnd + k)
            members[k].set_positions(git, rel)
            alone[k].set_positions(git, rel)
            if how in ("prepare", "both"):
                members[k].prepare()
            if how in ("pos write", "both"):
                members[k].write_pos_async(str(tmp_path / ("a%d" % k)), str(tmp_path / ("b%d" % k)), 0, 1.0)
            if how == "forces":
                members[k].berechne_WCA()
        b.run_steps(9)
        b.sync()
        for k, (a, m) in enumerate(zip(alone, members)):
            a.run_steps(9)
            (ga, ra), (gm, rm) = a.positions(), m.positions()
            assert np.array_equal(ga, gm) and np.array_equal(ra, rm), "member %d round %d" % (k, rnd)
    for m in members:
        m.write_wait()
    b.close()


def test_status_after_a_new_state():
    """bdk_batch_status right after a run-away member's new state: the flag is
    that of the new state."""
    print("case: batch status after a new state", flush=True)
    bad = [start(bdk.FP32, 1), start(bdk.FP32, 0)]
    bp, git, rel = make(bdk.FP32, 0)
    for _ in range(3):
        bad[1].set_positions(*overlapping(bp, git, rel))
        b = bdk.Batch(bad)
        b.run_steps(3)
        assert list(b.status()) == [bdk.OK, bdk.ERR_NONFINITE]
        bad[1].set_positions(git, rel)
        bad[1].prepare()
        assert list(b.status()) == [bdk.OK, bdk.OK]
        b.run_steps(3)
        b.sync()
        b.close()
