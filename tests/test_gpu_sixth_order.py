"""The 6th-order interpolation against the oracle on every level of the column,
where its vertical range changes (one-sided near the walls, none outside), on
columns shorter than its six levels, and at the horizontal edges of the domain.
Tolerance: 216 terms whose weights add up to at most 8 in magnitude, each with
some tens of roundings: 64 * 8 * 2^-53 = 6e-14, taken as 1e-12 of the largest
node value."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import Consts, DropletStep, Flags, Grid, Particles
from oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [3, 4, 5, 6, 7, 8, 13, 40])
@pytest.mark.parametrize("stretched", [False, True])
def test_every_level_matches_oracle(nnz, stretched):
    nx, ny = 9, 7
    grid = Grid.tanh_stretched(nx, ny, nnz, 0.02, 0.025, 0.005, 0.03) if stretched else Grid.uniform(nx, ny, nnz, 0.02, 0.025, 0.015)
    rng = np.random.default_rng(100 * nnz + stretched)
    fields = [m + rng.standard_normal((nx, ny, nnz + 2)) for m in (0.0, 0.0, 0.0, 300.0, 0.02)]
    x = np.concatenate([[0.0, grid.xl, grid.dx, np.nextafter(grid.xl, 0)], rng.uniform(0, grid.xl, 6)])
    y = np.concatenate([[0.0, grid.yl, grid.dy], rng.uniform(0, grid.yl, 7)])
    lev = np.concatenate([grid.zz, grid.z])
    z = np.concatenate([lev, lev + 1e-4, lev - 1e-4, rng.uniform(0, grid.zl, 200)])
    z = z[(z > 0) & (z < grid.zl)]
    pts = np.array([(a, b, h) for h in z for a, b in zip(rng.permutation(x), rng.permutation(y))])
    p = Particles.empty(len(pts))
    p["x"], p["y"], p["z"] = pts.T
    p["radius"], p["m_s"], p["kappa_s"], p["Tp"] = 1e-5, 1e-18, 1.2, 300.0
    flags = Flags(ilin=0)
    s = DropletStep(grid, Consts(), flags)
    s.set_fields(*fields)
    s.put(p)
    s.interp()
    got = s.get()
    ora = Oracle(grid, Consts(), flags)
    ora.set_fields(*fields)
    # the oracle indexes its arrays one row beyond their end for a droplet at
    # x = xl or y = yl exactly: there it interpolates at the periodic image 0
    want = p.copy()
    for c, end in (("x", grid.xl), ("y", grid.yl)):
        want[c] = np.where(want[c] >= end, 0.0, want[c])
    ora.interp(want.soa)
    for name, f in zip(("ufx", "ufy", "ufz", "Tf", "qinf"), fields):
        err = np.max(np.abs(got[name] - want[name]))
        assert err <= 1e-12 * np.max(np.abs(f)), (name, err)
    s.close()
