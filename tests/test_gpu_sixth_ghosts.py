"""The 6th-order interpolation reads the levels that the reference's lists name
and no others, with a weight or without one: a NaN in a ghost level (0 or nnz + 1)
of the fields reaches exactly the droplets that it reaches in the oracle, and
the others keep the values that they have with an ordinary ghost level."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import Consts, DropletStep, Flags, Grid, Particles
from oracle import Oracle

pytestmark = pytest.mark.gpu

NAMES = ("ufx", "ufy", "ufz", "Tf", "qinf")


@pytest.mark.parametrize("nnz", [3, 4, 5, 6, 7, 8, 9, 20])
@pytest.mark.parametrize("ghost", ["bottom", "top"])
def test_a_nan_in_a_ghost_level_stays_where_the_oracle_has_it(nnz, ghost):
    nx, ny = 7, 6
    grid = Grid.tanh_stretched(nx, ny, nnz, 0.02, 0.025, 0.005, 0.03)
    rng = np.random.default_rng(nnz)
    clean = [m + rng.standard_normal((nx, ny, nnz + 2)) for m in (0.0, 0.0, 0.0, 300.0, 0.02)]
    fields = [f.copy() for f in clean]
    for f in fields:
        f[:, :, 0 if ghost == "bottom" else nnz + 1] = np.nan
    lev = np.concatenate([grid.zz, grid.z])
    z = np.concatenate([lev, lev + 1e-4, lev - 1e-4, rng.uniform(0, grid.zl, 300)])
    z = z[(z > 0) & (z < grid.zl)]
    p = Particles.empty(z.size)
    p["x"], p["y"], p["z"] = rng.uniform(0, 0.99 * grid.xl, z.size), rng.uniform(0, 0.99 * grid.yl, z.size), z
    p["radius"], p["m_s"], p["kappa_s"], p["Tp"] = 1e-5, 1e-18, 1.2, 300.0
    flags = Flags(ilin=0)
    got = []
    for f in (clean, fields):
        s = DropletStep(grid, Consts(), flags)
        s.set_fields(*f)
        s.put(p)
        s.interp()
        got.append(s.get())
        s.close()
    ora = Oracle(grid, Consts(), flags)
    ora.set_fields(*fields)
    want = p.copy()
    ora.interp(want.soa)
    for name in NAMES:
        nan = np.isnan(want[name])
        assert np.array_equal(np.isnan(got[1][name]), nan), (name, np.flatnonzero(np.isnan(got[1][name]) != nan))
        assert np.array_equal(got[1][name][~nan], got[0][name][~nan]), name
