"""Device memory of a handle: uploads, read-back of positions and forces and
the observables of many particles use what bdk_create allocated, and what the
direct rho(k) sums of few particles need besides is given back when the
simulation goes on."""
import ctypes as C
import math

import numpy as np
import pytest

import bdk
from common import params
from helpers import to_git_rel

pytestmark = pytest.mark.gpu

SLACK = 4 << 20  # the runtime hands memory out in pieces of 2 MB


def free_memory():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def lattice(n, L):
    m = int(math.ceil(math.sqrt(n)))
    return (np.stack(np.meshgrid(np.arange(m), np.arange(m)), -1).reshape(-1, 2)[:n] + 0.5) * (L / m)


def uploads_and_reads(s, start):
    s.set_positions(*start)
    s.prepare()
    s.positions()
    s.berechne_WCA()
    s.berechne_kapkraefte()


def steps(s):
    s.run_steps(3)  # (the runtime holds some 16 MB per handle for the steps' graphs)


def observables(s):
    s.positions()
    for sp in (1, 2) if s.p.n2 else (1,):
        s.rho_k(sp)
    s.radial_profile(256, 0.5)
    s.density_stats(200)
    s.pair_correlation(64, 0.05)


def everything(s, start):
    uploads_and_reads(s, start)
    steps(s)
    observables(s)


@pytest.mark.parametrize("n1,n2", [(300000, 300000), (500000, 0), (90000, 90000)])
@pytest.mark.parametrize("prec", [bdk.FP32, bdk.FP64])
def test_reads_and_uploads_use_the_handles_memory(n1, n2, prec):
    print("case: memory of %d + %d particles, prec=%d" % (n1, n2, prec), flush=True)
    L = 1.6 * math.sqrt(n1 + n2)
    bp, _ = params(n1=n1, n2=n2, L=L, Z=512, precision=prec, lam=20.0)
    d = bdk.derived(bp)
    start = to_git_rel(lattice(n1 + n2, L), d["B"], d["nc"])
    warm = bdk.RunDynamik(bp)  # the runtime's own allocations (code, staging)
    everything(warm, start)
    warm.close()
    before = free_memory()
    s = bdk.RunDynamik(bp)
    created = free_memory()
    assert before - created <= bdk.footprint(bp) + 16 * SLACK
    uploads_and_reads(s, start)
    assert created - free_memory() <= SLACK
    steps(s)
    stepped = free_memory()
    observables(s)
    assert stepped - free_memory() <= SLACK
    s.ftrho_sums(1, 40, 4 * math.pi / L)  # (more than these particles' own arrays hold, for the smallest case)
    steps(s)
    assert stepped - free_memory() <= SLACK
    s.close()


def test_scratch_beyond_the_handle_is_given_back():
    print("case: scratch of the direct sums given back", flush=True)
    n, L = 2500, 100.0
    bp, _ = params(n1=n, n2=n, L=L, Z=64, precision=bdk.FP32)
    d = bdk.derived(bp)
    start = to_git_rel(lattice(2 * n, L), d["B"], d["nc"])
    sims = [bdk.RunDynamik(bp) for _ in range(8)]
    for s in sims:
        everything(s, start)
    sims[0].ftrho_sums(1, 120, 4 * math.pi / L)
    sims[0].run_steps(1)
    created = free_memory()
    dq = 4 * math.pi / L
    want = [v.copy() for v in sims[0].ftrho_sums(2, 120, dq)]
    for s in sims:
        s.ftrho_sums(1, 120, dq)
        s.prepare()
    assert created - free_memory() <= SLACK
    b = bdk.Batch(sims)
    b.run_steps(1)
    b.sync()
    stepped = free_memory()
    for s in sims:
        s.ftrho_sums(1, 120, dq)
    b.run_steps(1)
    b.sync()
    assert stepped - free_memory() <= SLACK
    b.close()
    # results do not depend on where the sums' scratch lies
    sims[1].set_positions(*start)
    sims[1].run_steps(4)
    sims[2].set_positions(*start)
    sims[2].run_steps(4)
    a = sims[1].ftrho_sums(2, 120, dq)
    sims[2].ftrho_sums(2, 7, dq)
    for u, v in zip(a, sims[2].ftrho_sums(2, 120, dq)):
        assert np.array_equal(u, v)
    assert len(want[0]) == len(a[0])
    for s in sims:
        s.close()
