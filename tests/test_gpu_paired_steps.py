"""Steps whose mesh and list stages share launches (small simulations) and
steps on two streams give the same run: a member of a batch always steps on
two streams, a lone handle of this size in pairs.  Every kind of mesh,
precision, force kernel and dt, the sizes on either side of a block, and a
step driven by calls between replayed ones."""
import numpy as np
import pytest

import bdk
from common import params
from helpers import to_git_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2,L,Z,scheme", [
    (1, 1, 8.0, 8, bdk.CIC), (40, 23, 12.0, 16, bdk.TSC), (33, 32, 15.0, 50, bdk.NGP), (700, 550, 60.0, 64, bdk.TSC),
    (900, 1100, 64.0, 128, bdk.CIC), (1500, 1001, 90.0, 250, bdk.TSC), (2000, 2000, 300.0, 384, bdk.TSC),
    (9000, 11000, 200.0, 512, bdk.TSC), (4000, 3000, 130.0, 600, bdk.CIC)])
@pytest.mark.parametrize("prec", [bdk.FP64, bdk.FP32, bdk.FP32_POS32K])
@pytest.mark.parametrize("travel,ratio", [(float("inf"), 1.0), (0.24, 1.0), (0.24, 1.1)])
def test_paired_steps_equal_two_streams(n1, n2, L, Z, scheme, prec, travel, ratio):
    print("case: paired steps n=%d+%d Z=%d prec=%d travel=%g ratio=%g" % (n1, n2, Z, prec, travel, ratio), flush=True)
    bp, _ = params(n1=n1, n2=n2, L=L, Z=Z, scheme=scheme, precision=prec, max_travel=travel, sigma11_12=ratio, seed=5)
    x = np.random.default_rng(n1).uniform(0.0, L, (n1 + n2, 2))
    d = bdk.derived(bp)
    start = to_git_rel(x, d["B"], d["nc"])
    lone, member = bdk.RunDynamik(bp), bdk.RunDynamik(bp)
    for s in (lone, member):
        s.set_positions(*start)
    b = bdk.Batch([member])
    b.run_steps(19)
    b.sync()
    lone.run_steps(9)
    lone.zeitschritt(1.0)
    lone.zeitschritt_debug(1.0)
    lone.run_steps(8)
    for a, m in zip(lone.positions(), member.positions()):
        assert np.array_equal(a, m)
    b.close()
    for s in (lone, member):
        s.close()
