"""Charge meshes of the tiled deposit (gridRoutinen.cpp:31-547) against the
textbook weights: meshes of one tile and of many with remainders, windows that
would cover the whole mesh, offsets beyond their list cell (the reference's
random start), every scheme.  Bounds: FP32 weights and charges are rounded a
few times at 2^-24 and truncated at 2^-31 of the largest charge; FP64 fixed
point is exact to 2^-40 and numpy's weights round a few times at 2^-53."""
import numpy as np
import pytest

import bdk
from common import params
from helpers import deposit_numpy, to_git_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Z,L", [(8, 30.0), (10, 5.0), (16, 61.0), (36, 20.0), (64, 40.0), (96, 300.0), (250, 120.0),
                                 (512, 350.0), (1024, 90.0)])
@pytest.mark.parametrize("scheme", [bdk.NGP, bdk.CIC, bdk.TSC])
@pytest.mark.parametrize("prec,tol", [(bdk.FP64, 1e-13), (bdk.FP32, 1e-6)])
def test_charge_mesh(Z, L, scheme, prec, tol):
    print("case: charge mesh Z=%d L=%g scheme=%d prec=%d" % (Z, L, scheme, prec), flush=True)
    n1, n2 = 700, 433
    bp, _ = params(n1=n1, n2=n2, L=L, Z=Z, scheme=scheme, lam=6.0, precision=prec, f2_f1=-0.7, seed=9)
    s = bdk.RunDynamik(bp)
    x = np.random.default_rng(Z).uniform(0.0, L, (n1 + n2, 2))
    for start in (to_git_rel(x, s.B, s.nc), bdk.MT(3).init_positions(bp)):
        s.set_positions(*start)
        s.berechne_kapkraefte()
        q = np.r_[np.ones(n1), np.full(n2, -0.7)]
        want = deposit_numpy(s.absolute(), q, Z, L / Z, scheme)
        got = s.mesh(bdk.MESH_RHO)
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    s.close()
