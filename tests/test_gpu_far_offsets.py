"""Charges and forces of particles far outside the cell they are listed in
(offsets of any size up to 1e9 are a state's to hold): cells below 0, the next
boxes on either side and several boxes away, with a last tile of one row of
list cells.  The reference truncates x / h toward zero (gridRoutinen.cpp:44,
154, 435), so below 0 the offset from the point's centre lies in (-1.5, -0.5);
the positions keep to [-1, -0.5], where both precisions' weights are the
textbook polynomials."""
import numpy as np
import pytest

import bdk
from common import params

pytestmark = pytest.mark.gpu


def weights(u, scheme):
    k = np.trunc(u)
    d = u - (k + 0.5)
    if scheme == bdk.NGP:
        w = np.stack([0 * d, 0 * d + 1, 0 * d], -1)
    elif scheme == bdk.CIC:
        w = np.stack([np.where(d < 0, -d, 0), 1 - np.abs(d), np.where(d < 0, 0, d)], -1)
    else:
        w = np.stack([0.5 * (0.5 - d) ** 2, 0.75 - d * d, 0.5 * (0.5 + d) ** 2], -1)
    return k.astype(np.int64), w


# mesh indices up to 3 Z = 1152, x / h rounded three times, and weights that
# change by at most 1.5 per mesh spacing: 1152 * 3 * 1.5 * 2^-53 = 6e-13 of a
# weight in FP64; FP32 weights, products and sums round about 30 times at 2^-24
TOL = {bdk.FP64: 2e-12, bdk.FP32: 4e-6}


@pytest.mark.parametrize("Z,L", [(10, 5.0), (36, 20.0), (90, 10.2), (250, 30.4), (384, 31.5), (256, 30.4)])
@pytest.mark.parametrize("scheme", [bdk.NGP, bdk.CIC, bdk.TSC])
@pytest.mark.parametrize("prec", [bdk.FP64, bdk.FP32])
def test_far_offsets(Z, L, scheme, prec):
    print("case: far offsets Z=%d L=%g scheme=%d prec=%d" % (Z, L, scheme, prec), flush=True)
    n1, n2, q2 = 60, 53, -0.7
    n = n1 + n2
    bp, _ = params(n1=n1, n2=n2, L=L, Z=Z, scheme=scheme, lam=2.0, precision=prec, f2_f1=q2, ngp_fix=1, seed=9)
    s = bdk.RunDynamik(bp)
    h = L / Z
    rng = np.random.default_rng(Z)
    cell = s.B / h
    below = lambda top: -(np.floor(rng.uniform(0, top, n)) + rng.uniform(0.05, 0.45, n))
    above = lambda lo, hi: np.floor(rng.uniform(lo, hi, n)) + rng.uniform(0.05, 0.95, n)
    inside = above(0, Z)
    far = [below(4 * cell), below(Z), above(Z, 2 * Z), below(3 * Z), above(2 * Z, 3 * Z)]
    for i, u in enumerate(far):
        for ux, uy in ((inside, u), (u, inside), (u, u[::-1])):
            x = np.stack([ux, uy], 1) * h
            # the in-box axis listed in its own cell, the far one in cell 0
            git = np.where((x >= 0) & (x < L), np.clip(np.floor(x / s.B), 0, s.nc - 1), 0).astype(np.int32)
            rel = x - git * s.B
            s.set_positions(git, rel)
            f = s.berechne_kapkraefte()
            x = git * s.B + rel
            (kx, wx), (ky, wy) = weights(x[:, 0] / h, scheme), weights(x[:, 1] / h, scheme)
            q = np.r_[np.ones(n1), np.full(n2, q2)]
            want, bound = np.zeros((Z, Z)), np.zeros((Z, Z))
            fx, fy = s.mesh(bdk.MESH_FX), s.mesh(bdk.MESH_FY)
            force, fb = np.zeros((n, 2)), 0.0
            for a in range(3):
                for b in range(3):
                    at, w = ((kx + a - 1) % Z, (ky + b - 1) % Z), wx[:, a] * wy[:, b]
                    np.add.at(want, at, q * w / (h * h))
                    np.add.at(bound, at, np.abs(q) / (h * h))
                    force += w[:, None] * np.stack([fx[at], fy[at]], 1)
            force[n1:] *= q2
            assert np.all(np.abs(s.mesh(bdk.MESH_RHO) - want) <= TOL[prec] * bound), "charges, case %d" % i
            top = max(np.abs(fx).max(), np.abs(fy).max())
            assert np.abs(f - force).max() <= 9 * TOL[prec] * top, "forces, case %d" % i
    s.close()
