"""Cells whose entries fill several waves: the list rebuild of a step ranks the
particles that stay in their cell by wave and adds the stayers of the whole
waves before (up to six of them here), beside movers into and out of the same
cells.  Against the oracle's trajectory with the same noise, and the lists
against the positions: every particle once, in its cell."""
import numpy as np
import pytest

import bdk
from common import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(63, 65, 1), (64, 64, 64), (129, 10, 200), (400, 1, 128), (70, 0, 450)])
@pytest.mark.parametrize("mode", ["alone", "ideal gas", "batch"])
def test_cells_of_several_waves(sizes, mode):
    print("case: dense cells %s %s" % (sizes, mode), flush=True)
    idgas, batch = int(mode == "ideal gas"), mode == "batch"
    L, nc = 8.0, 7
    B = L / nc
    rng = np.random.default_rng(sum(sizes))
    # the crowded cells side by side (the last two across the y edge), the rest spread
    cells = [(3, 5), (3, 6), (3, 0)]
    git = [c for c, n in zip(cells, sizes) for _ in range(n)]
    spread = [(int(a), int(b)) for a, b in rng.integers(0, nc, (90, 2))]
    git = np.array(git + spread, np.int32)
    git = git[rng.permutation(len(git))]
    rel = rng.uniform(0.0, B, (len(git), 2))
    n1 = len(git) // 2
    # a bounded pair force, so that some particles change cell in a step and none runs away
    g, o, _, _ = pair(git=git, rel=rel, n1=n1, n2=len(git) - n1, L=L, Z=16, scheme=bdk.CIC, lam=2.0, T=1.0,
                      dt_max=2e-3, max_pair_wca=1.0, idgas_only=idgas, precision=bdk.FP64, seed=5)
    assert g.nc == nc
    b = bdk.Batch([g]) if batch else None
    moved = 0
    for _ in range(6):
        before = g.positions()[0]
        if batch:
            b.run_steps(2)
            b.sync()
        else:
            g.run_steps(2)
        for _ in range(2):
            o.step(1.0)
        x, og = g.positions(), o.all_positions()
        moved += int((x[0] != before).any(1).sum())
        assert np.array_equal(x[0], og[0])
        assert np.abs(x[1] - og[1]).max() < 1e-9
        start, ids = g.cells()
        cell = x[0][:, 0] * nc + x[0][:, 1]
        assert np.array_equal(np.diff(start), np.bincount(cell, minlength=nc * nc))
        assert np.array_equal(np.sort(ids), np.arange(len(git)))
        assert np.array_equal(cell[ids], np.repeat(np.arange(nc * nc), np.diff(start)))
    assert moved > 20
    if b:
        b.close()
    g.close()
