"""The three FFT passes at every mesh size they are compiled for: the force
meshes against numpy's FP64 transform of the device's own charge mesh
(berechne_kapkraefte, dynamik_methoden.cpp:1180-1233: discrete symbols of
dm:585-593 and dm:1384-1394), and batches of mixed sizes under every number of
elements per thread against their members alone."""
import math

import numpy as np
import pytest

import bdk
from common import params
from helpers import to_git_rel

pytestmark = pytest.mark.gpu


def sim(Z, prec, seed, scheme=bdk.TSC):
    L = max(12.0, 0.6 * Z)
    n = 60 + 5 * Z
    bp, _ = params(n1=n, n2=n - 7, L=L, Z=Z, scheme=scheme, lam=6.0, precision=prec, seed=seed)
    x = np.random.default_rng(seed).uniform(0.0, L, (2 * n - 7, 2))
    d = bdk.derived(bp)
    s = bdk.RunDynamik(bp)
    s.set_positions(*to_git_rel(x, d["B"], d["nc"]))
    return s


@pytest.mark.parametrize("Z", [8, 16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 12, 250, 384, 600, 1400])
@pytest.mark.parametrize("prec,tol", [(bdk.FP64, 1e-12), (bdk.FP32, 1e-5)])
def test_force_meshes(Z, prec, tol):
    print("case: force meshes Z=%d prec=%d" % (Z, prec), flush=True)
    s = sim(Z, prec, 3)
    s.berechne_kapkraefte()
    rho = s.mesh(bdk.MESH_RHO)
    h, p = s.hmesh, s.p
    q = 2.0 * math.pi / p.L * ((np.arange(Z) + Z // 2) % Z - 0.5 * Z)
    sq, lap = p.kap * np.sin(q * h) / h, (2.0 * np.sin(0.5 * q * h) / h) ** 2
    G = 1.0 / (lap[:, None] + lap[None, :] + 1.0 / p.lam ** 2)
    if p.lam > 0.2 * p.L:
        G[0, 0] = 0.0
    S = np.fft.fft2(rho) * G * 1j
    for which, S1 in ((bdk.MESH_FX, S * sq[:, None]), (bdk.MESH_FY, S * sq[None, :])):
        want = np.fft.ifft2(S1).real
        got = s.mesh(which)
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    s.close()


@pytest.mark.parametrize("prec,sizes", [(bdk.FP32, (8, 64, 512, 1024, 2048, 96)), (bdk.FP64, (8, 32, 128, 1024, 50))])
@pytest.mark.parametrize("ept", [8, 16, 32])
def test_mixed_batch_equals_members_alone(prec, sizes, ept):
    print("case: mixed batch prec=%d ept=%d" % (prec, ept), flush=True)
    alone, members = [sim(Z, prec, 5) for Z in sizes], [sim(Z, prec, 5) for Z in sizes]
    b = bdk.Batch(members)
    b.set_tuning(ept_r2c=ept, ept_col=ept, ept_c2r=ept)
    b.run_steps(2)
    b.sync()
    for a, m in zip(alone, members):
        a.run_steps(2)
        assert np.array_equal(a.mesh(bdk.MESH_FX), m.mesh(bdk.MESH_FX))
        assert np.array_equal(a.absolute(), m.absolute())
    b.close()
    for s in alone + members:
        s.close()
