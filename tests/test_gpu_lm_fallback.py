"""The two forms of the Levenberg-Marquardt fallback, one evaluation of the
equations per iteration (the serving step, every FP64 step) and two (the mixed
step of the library), give the same bits: a population of which a fifth falls
back is served and stepped, and both must agree, counters included."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import (MODE_BE, PREC_FP64, PREC_MIXED, SERVE_IN, SERVE_OUT, Consts, DropletStep, Flags, ServeLoop,
                      synth)

from .helpers import mixed_droplets, small_grid

pytestmark = pytest.mark.gpu

COUNTERS = ("num100", "numimpos", "actnum", "denum", "gn_iters", "lm_iters", "solves")


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("n", [1, 63, 65, 20_000])
def test_served_population_equals_plain(prec, n):
    rng = np.random.default_rng(11)
    grid, consts = small_grid("uniform"), Consts(dt=0.05, radius_init=5e-6)
    s = DropletStep(grid, consts, Flags())
    s.set_fields(*synth.make_fields(grid, consts, rng, T0=300.0, T_sd=0.1, rh_uniform=(80, 120)))
    p = mixed_droplets(grid, rng, n)
    s.put(p)
    s.interp(set_vp=True, set_tp=True)
    s.crit_radius()
    s.counters(reset=True)
    s.step(MODE_BE, prec, nsteps=2, it0=2)
    plain, c = s.get(), s.counters()
    if n > 1000:
        assert c["num100"] > n // 8, c
    loop = ServeLoop(s, 1 << 28, steps=2, precision=prec)
    inp = np.ascontiguousarray(np.stack([p[k] for k in SERVE_IN]))
    out, mult = np.empty((len(SERVE_OUT), n)), np.empty(n, dtype=np.int64)
    loop.wait(loop.submit(inp, p.mult, out, mult))
    for i, k in enumerate(SERVE_OUT):
        assert np.array_equal(out[i], plain[k]), k
    newton = loop.close()["newton"]
    assert [newton[k] for k in COUNTERS] == [c[k] for k in COUNTERS]
    s.close()
