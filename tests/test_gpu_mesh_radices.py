"""Mesh passes planned from radices 2 to 14 (sizes that are not powers of two),
at sizes that take every radix as the first, a middle and the last pass, with
two to four passes and rows of few and of 128 threads, and sizes beside their
range (10 and 14: a prime half; 1500: rows too long).  Against numpy's FP64
transform, and in batches against the members alone."""
import pytest

import bdk
import test_gpu_fft_sizes as sizes

pytestmark = pytest.mark.gpu

MESHES = [10, 12, 14, 18, 20, 24, 28, 36, 42, 50, 54, 70, 90, 98, 126, 144, 162, 192, 210, 300, 360, 432, 490, 640,
          686, 768, 810, 864, 882, 900, 960, 972, 1000, 1008, 1500]


@pytest.mark.parametrize("Z", MESHES)
@pytest.mark.parametrize("prec,tol", [(bdk.FP64, 1e-12), (bdk.FP32, 1e-5)])
def test_force_meshes(Z, prec, tol):
    sizes.test_force_meshes(Z, prec, tol)


@pytest.mark.parametrize("prec", [bdk.FP64, bdk.FP32])
@pytest.mark.parametrize("meshes", [(10, 12, 18, 64, 90, 126), (300, 250, 1500, 384), (1000, 686, 14, 144)])
def test_batches_equal_members_alone(prec, meshes):
    sizes.test_mixed_batch_equals_members_alone(prec, meshes, 8)
