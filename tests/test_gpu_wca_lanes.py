"""FP64 WCA forces, four lanes per particle: numbers of particles around a
block (64), boxes of 3 cells (every neighbour an image) and more, unequal
species, against the oracle (dynamik_methoden.cpp:617-1059).  Uncorrelated
positions: pairs at all distances, many at the force cap."""
import numpy as np
import pytest

import bdk
from common import params
from helpers import rel_rms, to_git_rel
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [3.4, 4.6, 7.0, 30.0])
@pytest.mark.parametrize("n1,n2", [(1, 0), (1, 1), (15, 2), (63, 0), (40, 24), (33, 32), (150, 107)])
@pytest.mark.parametrize("ratios", [{}, dict(sigma11_22=1.2, sigma11_12=1.1, eps22_11=0.7, eps12_11=0.9)])
def test_fp64_wca_against_oracle(L, n1, n2, ratios):
    print("case: FP64 WCA L=%g n=%d+%d" % (L, n1, n2), flush=True)
    bp, op = params(n1=n1, n2=n2, L=L, Z=16, precision=bdk.FP64, **ratios)
    x = np.random.default_rng(n1 + 7).uniform(0.0, L, (n1 + n2, 2))
    d = bdk.derived(bp)
    git, rel = to_git_rel(x, d["B"], d["nc"])
    s, o = bdk.RunDynamik(bp), O.Oracle(op)
    s.set_positions(git, rel)
    o.set_all(git, rel)
    got, want = s.berechne_WCA(), o.wca()
    if np.any(want):
        assert rel_rms(got, want) <= 1e-12
    else:
        assert not np.any(got)
    s.close()
    o.close()
