"""The scan of the u-cell counts on both sides of the line between its two forms
(1400 tiles of 8192 cells): a grid that fills 1400 tiles to the last cell, the next
larger ones, and one far beyond, against numpy."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import Consts, DropletStep, Flags, Grid, Particles

pytestmark = pytest.mark.gpu

# nodes (nnx+1, nny+1, nnz+1): 1394.5, 1400, 1402, 1406.25 and 3372.8 tiles
NODES = [(224, 200, 255), (224, 200, 256), (216, 252, 211), (225, 200, 256), (300, 300, 307)]


@pytest.mark.parametrize("nodes", NODES)
def test_bin_offsets(nodes):
    nx, ny, nz = (v - 1 for v in nodes)
    g = Grid.uniform(nx, ny, nz, 0.01, 0.01, 0.01)
    s = DropletStep(g, Consts(), Flags())
    rng = np.random.default_rng(nx)
    n = 50_000
    p = Particles.empty(n)
    # a third in the first columns, a third in the last, a third everywhere
    x = rng.uniform(0, g.xl, n)
    x[::3], x[1::3] = x[::3] * 0.01, g.xl - x[1::3] * 0.01
    p["x"], p["y"], p["z"] = x, rng.uniform(0, g.yl, n), rng.uniform(0, g.zl, n)
    p["radius"] = 1e-5
    s.put(p)
    cell, counts, offsets, perm = s.bin()
    key = cell[:, 2] + (g.nnz + 1) * ((cell[:, 1] - 1) + (g.nny + 1) * (cell[:, 0] - 1).astype(np.int64))
    want = np.bincount(key, minlength=counts.size)
    assert np.array_equal(counts, want)
    assert np.array_equal(offsets, np.concatenate([[0], np.cumsum(want)]))
    assert np.array_equal(perm, np.argsort(key, kind="stable"))
    s.close()
