"""Read-back of positions and forces in id order, at the sizes where its route
changes: results written straight to the host's staging up to 4096 particles,
by a second kernel up to 4 MB (174,751 positions, 262,144 forces), copied to
the caller's memory above.  Positions come back as they were set; particles
2k and 2k + 1 repel at a distance that grows with k, so the force tells whose
it is."""
import math

import numpy as np
import pytest

import bdk
from common import params
from helpers import to_git_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1", [2, 4094, 4096, 4098, 174748, 174754, 262144, 262146])
@pytest.mark.parametrize("n2", [0, 2])
def test_read_back_in_id_order(n1, n2):
    print("case: read-back of %d + %d particles" % (n1, n2), flush=True)
    pairs = (n1 + n2) // 2
    m = max(2, math.isqrt(pairs - 1) + 1)
    bp, _ = params(n1=n1, n2=n2, L=3.0 * m, Z=64, precision=bdk.FP64)
    k = np.arange(pairs)
    gap = 0.95 + 0.1 * k / pairs  # inside the cutoff 2^(1/6), below the force cap
    x = np.empty((pairs, 2, 2))
    x[:, :, 0] = (3.0 * (k % m) + 1.0)[:, None]
    x[:, :, 1] = (3.0 * (k // m) + 1.0)[:, None]
    x[:, 1, 0] += gap
    order = np.random.default_rng(n1 + n2).permutation(pairs)  # ids not in storage order
    x, gap = x[order].reshape(-1, 2), gap[order]
    d = bdk.derived(bp)
    git, rel = to_git_rel(x, d["B"], d["nc"])
    s = bdk.RunDynamik(bp)
    s.set_positions(git, rel)
    g, r = s.positions()
    assert np.array_equal(g, git) and np.array_equal(r, rel)
    f = s.berechne_WCA().reshape(pairs, 2, 2)
    assert np.array_equal(f[:, 0], -f[:, 1]) and not np.any(f[:, :, 1])
    push = f[:, 1, 0][np.argsort(gap)]
    assert np.all(push > 0.0) and np.all(np.diff(push) < 0.0)
    s.close()


@pytest.mark.parametrize("precision", [bdk.FP64, bdk.FP32, bdk.FP32_POS32, bdk.FP32_POS32K])
@pytest.mark.parametrize("n1,n2", [(1, 0), (255, 2), (3000, 1000), (150000, 60000)])
def test_a_state_replaced_before_it_was_waited_for(precision, n1, n2):
    print("case: replaced state, %d + %d particles, precision %d" % (n1, n2, precision), flush=True)
    n, L = n1 + n2, max(8.0, 1.6 * math.sqrt(n1 + n2))
    bp, _ = params(n1=n1, n2=n2, L=L, Z=64, precision=precision)
    d, rng = bdk.derived(bp), np.random.default_rng(n)
    states = [to_git_rel(rng.uniform(0.0, L, (n, 2)), d["B"], d["nc"]) for _ in range(3)]
    s, fresh = bdk.RunDynamik(bp), bdk.RunDynamik(bp)
    for git, rel in states:
        s.set_positions(git, rel)
        s.prepare()  # enqueues the lists and forces
    fresh.set_positions(*states[-1])
    for got, want in zip(s.positions() + s.cells(), fresh.positions() + fresh.cells()):
        assert np.array_equal(got, want)
    assert np.array_equal(s.positions()[0], states[-1][0])
    assert np.array_equal(s.berechne_WCA(), fresh.berechne_WCA())
    assert np.array_equal(s.berechne_kapkraefte(), fresh.berechne_kapkraefte())
    s.close()
    fresh.close()
