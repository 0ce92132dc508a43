"""Mixed backward-Euler steps on both sides of the size from which fallback solves
evaluate twice: droplet i of a population just above it ends with the bits that it
gets in the populations at and below it, with a fifth of the solves falling
back, in calls of two steps and of many (residence times settled at their end)."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import COLUMNS, MODE_BE, PREC_MIXED, Consts, DropletStep, Flags, Particles, synth

from .helpers import mixed_droplets, small_grid

pytestmark = pytest.mark.gpu

LINE = 3 * 1024 * 64


@pytest.mark.parametrize("nsteps", [2, 12])
def test_same_bits_on_both_sides(nsteps):
    rng = np.random.default_rng(12)
    grid, consts = small_grid(), Consts(dt=0.05, radius_init=5e-6)
    s = DropletStep(grid, consts, Flags())
    s.set_fields(*synth.make_fields(grid, consts, rng, T0=300.0, T_sd=0.1, rh_uniform=(80, 120)))
    p = mixed_droplets(grid, rng, LINE + 1)
    want = None
    for n in (LINE + 1, LINE, 77):
        s.put(Particles(p.soa[:, :n].copy(), p.mult[:n].copy(), p.pidx[:n].copy(), p.procidx[:n].copy()))
        s.interp(set_vp=True, set_tp=True)
        s.crit_radius()
        s.counters(reset=True)
        s.step(MODE_BE, PREC_MIXED, nsteps=nsteps, it0=2)
        got = s.get()
        if want is None:
            want = got
            assert s.counters()["num100"] > n // 8
        for c in COLUMNS:
            assert np.array_equal(got[c].view(np.uint64), want[c][:n].copy().view(np.uint64)), (c, n)
    s.close()
