"""The direct rho(k) sums (auswertung.cpp:307-360) against extended precision,
for every tile of index pairs (8, 16, 32 a side, and several) and both routes
of the species-1 y coordinate.

Bound on the relative error of all sums together.  A factor's angle is reduced
without rounding and its sine and cosine are then good to about 3 units of
2^-53, a product of two to 7 and a little; over N independent terms that is
8 * 2^-53 sqrt(N / 3) against sums of size sqrt(N / 2): 7e-16.  Adding up in
chains of at most some 130 rounds by 2^-53 of the running sum each time,
independently: sqrt(130 / 3) * 2^-53 = 7e-16.  Together 1e-15, and a factor of
two.  (A sum of cos(dq (x i + y j)) in FP64 is off by 2e-14 at 70 bins.)"""
import math

import numpy as np
import pytest

import bdk
from test_gpu_obs_shapes import random_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2", [(70, 3000), (2500, 1200)])
@pytest.mark.parametrize("qbins", [2, 8, 9, 16, 17, 33, 70])
@pytest.mark.parametrize("fix", [0, 1])
def test_sums_against_extended_precision(n1, n2, qbins, fix):
    print("case: ftrho against extended precision n=%d+%d qbins=%d fix=%d" % (n1, n2, qbins, fix), flush=True)
    assert np.finfo(np.longdouble).eps < 2.0 ** -60
    L = 90.0
    s = random_sim(n1, n2, L, 43 + n1, ftrho_fix=fix)
    g, r = s.positions()
    x = g * s.B + r
    if not fix:
        x[:n1, 1] = g[:n1, 1] * s.B + r[:n1, 0]
    dq = 4.0 * math.pi / L
    pairs = np.array([(i, j) for i in range(qbins) for j in range(qbins) if i * i + j * j <= qbins * qbins], np.longdouble)
    for sp, xs in ((1, x[:n1]), (2, x[n1:])):
        re, im = s.ftrho_sums(sp, qbins, dq)
        a = np.longdouble(dq) * (pairs @ xs.T.astype(np.longdouble))
        want = np.r_[np.cos(a).sum(1), np.sin(a).sum(1)]
        err = np.r_[re, im] - want
        rel = float(np.sqrt((err * err).sum() / (want * want).sum()))
        print("species %d: %.2e" % (sp, rel), flush=True)
        assert rel <= 2e-15
    s.close()
