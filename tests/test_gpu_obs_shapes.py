"""Device observables at the sizes where their kernels can go wrong: edges of
tiles, remainders, the smallest inputs, both sides of each choice of kernel."""
import math

import numpy as np
import pytest

import bdk
from common import params
from helpers import (density_stats_ref, pair_correlation_ref, radial_profile_ref, rho_k_ref, to_git_rel,
                     tsc_snapshot_ref)

pytestmark = pytest.mark.gpu


def random_sim(n1, n2, L, seed, **kw):
    """Uncorrelated positions (pairs at every distance down to ~0)."""
    bp, _ = params(n1=n1, n2=n2, L=L, seed=seed, **dict(dict(Z=64, precision=bdk.FP64), **kw))
    x = np.random.default_rng(seed).uniform(0.0, L, (n1 + n2, 2))
    d = bdk.derived(bp)
    s = bdk.RunDynamik(bp)
    s.set_positions(*to_git_rel(x, d["B"], d["nc"]))
    return s


@pytest.mark.parametrize("n1,n2", [(2, 2), (31, 33), (300, 212), (511, 2), (500, 77), (525, 499), (1100, 1013)])
@pytest.mark.parametrize("rmax,nbins", [(2.0, 7), (8.5, 400), (13.4, 61), (15.2, 4096), (40.0, 33)])
def test_pair_counts_at_tile_edges(n1, n2, rmax, nbins):
    """Both kernels of the pair histogram (cells within the range, all pairs)
    against every pair by brute force, as whole counts: numbers of particles
    around the tiles of 64 and 1024, ranges up to and across half the box
    (nc = 27: 12 cells are the last range that does not cover it)."""
    print("case: pair counts n=%d+%d rmax=%g nbins=%d" % (n1, n2, rmax, nbins), flush=True)
    L = 30.5
    s = random_sim(n1, n2, L, 11 + n1)
    assert s.nc == 27
    dr = rmax / nbins
    g = s.pair_correlation(nbins, dr)
    noalloc = s.pair_correlation_noalloc(nbins, dr)
    x = s.absolute()
    want = pair_correlation_ref(x[:n1], x[n1:], L, nbins, dr)
    for got, same, ref in zip(g, noalloc, want):
        assert np.allclose(got, ref, rtol=1e-12, atol=0)
        assert np.array_equal(got, same)
    s.close()


@pytest.mark.parametrize("Z", [8, 10, 64, 250, 512])
@pytest.mark.parametrize("ratio,nbins", [(0.5, None), (0.5, 1), (1.0, 4), (0.37, 200), (2.5, 3)])
def test_rho_k_shells(Z, ratio, nbins):
    """Shell sums and lattice points per shell (one thread per shell and
    column) against the full plane: the smallest meshes, an odd Z/2, one
    shell, shells wider and narrower than a mesh mode, more shells than the
    plane holds."""
    nb = nbins or int(0.5 * Z * ratio)
    print("case: rho(k) shells Z=%d ratio=%g nbins=%d" % (Z, ratio, nb), flush=True)
    n1, n2, L = 300, 211, 30.5
    s = random_sim(n1, n2, L, 17, Z=Z, scheme=bdk.TSC)
    x = s.absolute()
    # the Nyquist column of an odd Z/2 enters with the sign of an even one
    top = nb if Z % 4 == 0 else min(nb, int(ratio * (Z // 2) + 0.5))
    for sp, xs in ((1, x[:n1]), (2, x[n1:])):
        re, im = s.rho_k(sp, ratio, nb)
        want = rho_k_ref(xs, L, Z, bdk.TSC, ratio, nb)
        assert np.abs(re - want)[:top].max() < 1e-11 * n1
        assert not im.any()
    s.close()


@pytest.mark.parametrize("n1,n2", [(1, 1), (130, 126), (1100, 949), (2048, 1), (9000, 8000)])
@pytest.mark.parametrize("nbins,dr", [(1, 3.0), (60, 0.5), (2048, 0.01), (2049, 0.01)])
def test_radial_profile_at_block_edges(n1, n2, nbins, dr):
    """One block and several, species of one particle, and both homes of the
    histogram (LDS up to 2048 bins)."""
    print("case: radial profile n=%d+%d nbins=%d" % (n1, n2, nbins), flush=True)
    L = 60.5
    s = random_sim(n1, n2, L, 23 + n1)
    cen, prof = s.radial_profile(nbins, dr)
    x = s.absolute()
    cref, pref = radial_profile_ref(x[:n1], x[n1:], L, nbins, dr)
    assert np.allclose(cen, cref, rtol=0, atol=1e-9 * L)
    # whole counts: a value within rounding of a bin edge may differ
    assert np.isclose(prof, pref, rtol=1e-12, atol=0).mean() > 0.999
    ring = np.pi * dr * dr * (2 * np.arange(nbins) + 1)
    assert np.allclose((prof * ring).sum(1), L * L, rtol=1e-12)
    s.close()


@pytest.mark.parametrize("m", [1, 2, 3, 5, 31, 32, 33, 64, 97, 300])
@pytest.mark.parametrize("outside", [False, True])
def test_snapshot_tiles(m, outside):
    """Tiles of the snapshot grid: one cell to several tiles with remainders,
    grid cells wider and narrower than list cells, list ranges that wrap, and
    (outside) offsets beyond their list cell, as the reference's random start
    leaves them.  Same bound as the whole-grid test: every contribution is
    rounded to 2^-41 of a weight."""
    print("case: snapshot tiles m=%d outside=%d" % (m, outside), flush=True)
    n1, n2, L = 900, 700, 61.3
    s = random_sim(n1, n2, L, 29)
    if outside:
        s.set_positions(*bdk.MT(31).init_positions(s.p))
        assert s.positions()[1].max() > s.B
    r1, r2 = s.density_grid(m)
    x = s.absolute()
    w1, w2 = tsc_snapshot_ref(x[:n1], x[n1:], L, m)
    w = L / m
    for got, ref, xs in ((r1, w1, x[:n1]), (r2, w2, x[n1:])):
        k = np.floor(xs / w).astype(np.int64)
        cnt = np.zeros((m, m))
        for a in (-1, 0, 1):
            for b in (-1, 0, 1):
                np.add.at(cnt, ((k[:, 0] + a) % m, (k[:, 1] + b) % m), 1.0)
        assert np.all(np.abs(got - ref) <= cnt * (2.0 ** -41 + 1e-15) / (w * w))
    th, dth = (0.1, 0.2, 0.5), (0.1, 0.2, 0.5, 0.99)
    for nbins, dbin in ((100, 0.01), (1, 1.0), (4096, 0.001)):
        hist, over = s.density_stats(m, nbins, dbin, th, dth)
        hr, orf = density_stats_ref(r1, r2, nbins, dbin, th, dth)
        assert np.array_equal(hist, hr) and np.array_equal(over, orf)
    s.close()


@pytest.mark.parametrize("n1,n2", [(1, 1), (31, 33), (257, 64), (900, 4000)])
@pytest.mark.parametrize("qbins", [1, 16, 17, 32, 33, 70])
def test_ftrho_tiles(n1, n2, qbins):
    """Tiles of 32 x 32 index pairs with remainders, species of fewer and more
    particles than a batch of 32, list parts without the species.  Bound: the
    numpy side rounds each angle (up to 2 pi 2 qbins sqrt 2) three times."""
    print("case: ftrho tiles n=%d+%d qbins=%d" % (n1, n2, qbins), flush=True)
    L = 90.0
    s = random_sim(n1, n2, L, 37 + n1, ftrho_fix=1)
    x, dq = s.absolute(), 4.0 * np.pi / L
    pairs = np.array([(i, j) for i in range(qbins) for j in range(qbins) if i * i + j * j <= qbins * qbins])
    for sp, xs in ((1, x[:n1]), (2, x[n1:])):
        re, im = s.ftrho_sums(sp, qbins, dq)
        assert len(re) == len(pairs)
        a = dq * (pairs @ xs.T)
        tol = len(xs) * (4 * math.pi * qbins * math.sqrt(2.0) * 3 * 2.0 ** -53 + 1e-15)
        assert np.abs(re - np.cos(a).sum(1)).max() <= tol and np.abs(im - np.sin(a).sum(1)).max() <= tol
        assert re[0] == len(xs) and im[0] == 0.0
    s.close()
