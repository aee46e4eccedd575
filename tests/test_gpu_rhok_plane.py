"""rho(k) of every shell (auswertung.cpp:529-626) against numpy's transform of
the full plane: meshes whose half size is odd, where the Nyquist column's sign
differs from the first column's, and the column kernels of every size and
precision (FP32 from 1024 points on has 16 points per thread, FP64 rows of 1024
points and more take several waves).

Bound.  A transform of Z^2 points rounds at most some 6 times per factor of 2,
so the spectrum is off by dF with |dF|_2 <= 6 log2(Z^2) eps Z |rho|_2, and a
shell's mean over cnt points by |dF|_2 / sqrt(cnt) (Cauchy-Schwarz), times
L^2/Z^2.  The deposited weights are off by a few eps each: N 8 eps at most in
any sum over the particles."""
import math

import numpy as np
import pytest

import bdk
from helpers import deposit_numpy, rho_k_ref
from test_gpu_obs_shapes import random_sim

pytestmark = pytest.mark.gpu


def check(Z, prec, ratio, nb, scheme=bdk.TSC):
    print("case: rho(k) over the plane Z=%d prec=%d ratio=%g nbins=%d" % (Z, prec, ratio, nb), flush=True)
    n1, n2, L = 300, 211, 30.5 if Z <= 2048 else 90.5  # (a mesh finer than 84 points per list cell is refused)
    s = random_sim(n1, n2, L, 41, Z=Z, scheme=scheme, precision=prec)
    x = s.absolute()
    eps = 2.0 ** -53 if prec == bdk.FP64 else 2.0 ** -24
    k = np.abs(((np.arange(Z) + Z // 2) % Z) - Z // 2).astype(float)
    b = (ratio * np.sqrt(k[:, None] ** 2 + k[None, :] ** 2) + 0.5).astype(np.int64).ravel()
    cnt = np.maximum(np.bincount(b, minlength=nb)[:nb], 1)
    for sp, xs in ((1, x[:n1]), (2, x[n1:])):
        rho = np.linalg.norm(deposit_numpy(xs, np.ones(len(xs)), Z, L / Z, scheme))
        re, im = s.rho_k(sp, ratio, nb)
        tol = (L / Z) ** 2 * 6 * 2 * math.log2(Z) * eps * Z * rho / np.sqrt(cnt) + len(xs) * 8 * eps
        if prec == bdk.FP64:  # numpy's own rounding, and x / h of numpy and kernel a few units apart
            tol = 2 * tol + len(xs) * 8 * Z * eps
        assert np.all(np.abs(re - rho_k_ref(xs, L, Z, scheme, ratio, nb)) <= tol)
        assert not im.any()
    s.close()


@pytest.mark.parametrize("Z", [10, 14, 18, 30, 90, 126, 150, 162, 210, 250, 270])
@pytest.mark.parametrize("prec", [bdk.FP32, bdk.FP64])
def test_odd_half_sizes(Z, prec):
    for ratio, nb in ((0.5, Z), (1.0, Z), (0.5, int(0.25 * Z)), (2.5, 3 * Z)):
        check(Z, prec, ratio, nb)


@pytest.mark.parametrize("Z,prec", [(8, bdk.FP32), (64, bdk.FP32), (512, bdk.FP32), (1024, bdk.FP32), (2048, bdk.FP32),
                                    (4096, bdk.FP32), (384, bdk.FP32), (1000, bdk.FP32), (2000, bdk.FP32),
                                    (1024, bdk.FP64), (2048, bdk.FP64), (4096, bdk.FP64), (2000, bdk.FP64)])
def test_column_kernels(Z, prec):
    check(Z, prec, 0.5, int(0.36 * Z))
