"""The scan of the u-cell counts: its tiles (8192 cells) and its two forms, one
workgroup per tile adding up the tiles before it (up to 16384 tiles) and the
three-pass form beyond, against numpy on cells and droplets where a tile ends,
a tile is left empty, or only the last tile holds anything."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import Consts, DropletStep, Flags, Grid, Particles

pytestmark = pytest.mark.gpu

# (nnx+1)(nny+1)(nnz+1) cells: less than a tile, exactly one, one over, several with a remainder, above 16384 tiles
GRIDS = [(7, 5, 9), (31, 15, 15), (2, 682, 3), (60, 50, 70), (520, 520, 500)]


@pytest.mark.parametrize("dims", GRIDS)
def test_bin_offsets(dims):
    nx, ny, nz = dims
    g = Grid.uniform(nx, ny, max(nz, 3), 0.01, 0.01, 0.01)
    s = DropletStep(g, Consts(), Flags())
    rng = np.random.default_rng(nx)
    n = 20_000
    p = Particles.empty(n)
    # half of the droplets in the first cell columns, half in the last: empty tiles between
    p["x"] = np.where(np.arange(n) % 2 == 0, rng.uniform(0, 0.03, n) % g.xl, g.xl - rng.uniform(1e-6, 0.02, n) % g.xl)
    p["y"] = rng.uniform(0, g.yl, n)
    p["z"] = rng.uniform(0, g.zl, n)
    p["radius"] = 1e-5
    s.put(p)
    cell, counts, offsets, perm = s.bin()
    key = cell[:, 2] + (g.nnz + 1) * ((cell[:, 1] - 1) + (g.nny + 1) * (cell[:, 0] - 1).astype(np.int64))
    want = np.bincount(key, minlength=counts.size)
    assert np.array_equal(counts, want)
    assert np.array_equal(offsets, np.concatenate([[0], np.cumsum(want)]))
    assert np.array_equal(perm, np.argsort(key, kind="stable"))
    s.close()
