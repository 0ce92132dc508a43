"""The FP64 backward-Euler solve inside and outside the range of values for
which it divides through reciprocals.  Ordinary droplets (inside) and a constant
outside it (no surface tension): one step against the oracle, counters exact,
within the bounds of the FP64 parity tests.  Droplets outside it (too little salt,
too small, too cold or hot) among ordinary ones: every droplet ends with the bits
that it gets in company of its own kind, whichever of the two forms its wave
runs."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import COLUMNS, PREC_FP64, Consts, DropletStep, Flags, Particles, synth
from oracle import Oracle

from .helpers import init_state, mixed_droplets, small_grid
from .test_gpu_parity import COUNTERS, compare

pytestmark = pytest.mark.gpu


def population(gam, n):
    rng = np.random.default_rng(21)
    grid, consts, flags = small_grid(), Consts(dt=5e-4, radius_init=5e-6, Gam=gam), Flags()
    ora = Oracle(grid, consts, flags)
    fields = synth.make_fields(grid, consts, rng, T0=300.0, T_sd=0.1, rh_uniform=(99.7, 100.5))
    ora.set_fields(*fields)
    p = mixed_droplets(grid, rng, n)
    init_state(ora, p)
    s = DropletStep(grid, consts, flags)
    s.set_fields(*fields)
    return s, ora, p


def stepped(s, p):
    s.put(p)
    s.counters(reset=True)
    s.particle_update_BE(it=2, precision=PREC_FP64)
    return s.get(), s.counters()


@pytest.mark.parametrize("gam", [7.28e-2, 0.0])
def test_ordinary_droplets_match_the_oracle(gam):
    s, ora, p = population(gam, 500)
    got, cnt = stepped(s, p)
    want = p.copy()
    cnt_o = ora.update_be(want.soa, 2)
    assert {k: cnt[k] for k in COUNTERS} == {k: cnt_o[k] for k in COUNTERS}
    bad = compare(got, want, ["x", "y", "z", "vx", "vy", "vz", "Tf", "qinf", "Tp", "radius", "qstar"])
    assert not bad, bad
    s.close()


@pytest.mark.parametrize("column,value", [("m_s", 0.0), ("m_s", 1e-47), ("radius", 8e-13), ("Tp", 1e-13), ("Tp", 1e13)])
def test_mixed_company(column, value):
    s, _, p = population(7.28e-2, 500)
    odd = np.arange(500) % 7 == 0
    p[column][odd] = value
    both, _ = stepped(s, p)
    for pick in (odd, ~odd):
        q = Particles(p.soa[:, pick].copy(), p.mult[pick].copy(), p.pidx[pick].copy(), p.procidx[pick].copy())
        alone, _ = stepped(s, q)
        for c in COLUMNS:
            assert np.array_equal(alone[c].view(np.uint64), both[c][pick].copy().view(np.uint64)), (c, value)
    s.close()
