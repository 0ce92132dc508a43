"""The two forms of the Levenberg-Marquardt fallback in mixed precision: above
kKeepMax droplets the library's step evaluates the equations twice per iteration,
the serving step once whatever its size.  A population just above that line, a fifth
of which falls back, gives the same bits and counters served and stepped."""
from __future__ import annotations

import os
import re

import numpy as np
import pytest

import ntlp_amd
from ntlp_amd import (MODE_BE, PREC_MIXED, SERVE_BYTES_PER_DROPLET, SERVE_IN, SERVE_OUT, Consts, DropletStep, Flags,
                      ServeLoop, synth)

from .helpers import mixed_droplets, small_grid

pytestmark = pytest.mark.gpu

COUNTERS = ("num100", "numimpos", "actnum", "denum", "gn_iters", "lm_iters", "solves")


def keep_max() -> int:
    with open(os.path.join(os.path.dirname(ntlp_amd.__file__), "csrc", "ntlp_gpu.hip")) as f:
        factors = re.search(r"constexpr int64_t kKeepMax = ([\d *]+);", f.read()).group(1)
    return int(np.prod([int(k) for k in factors.split("*")]))


@pytest.mark.parametrize("above", [1, 64])
def test_served_equals_stepped_above_the_line(above):
    n = keep_max() + above
    rng = np.random.default_rng(13)
    grid, consts = small_grid("uniform"), Consts(dt=0.05, radius_init=5e-6)
    s = DropletStep(grid, consts, Flags())
    s.set_fields(*synth.make_fields(grid, consts, rng, T0=300.0, T_sd=0.1, rh_uniform=(80, 120)))
    p = mixed_droplets(grid, rng, n)
    s.put(p)
    s.interp(set_vp=True, set_tp=True)
    s.crit_radius()
    s.counters(reset=True)
    s.step(MODE_BE, PREC_MIXED, nsteps=2, it0=2)
    plain, c = s.get(), s.counters()
    assert c["num100"] > n // 8, c
    loop = ServeLoop(s, 2 * n * SERVE_BYTES_PER_DROPLET, steps=2, precision=PREC_MIXED)
    inp = np.ascontiguousarray(np.stack([p[k] for k in SERVE_IN]))
    out, mult = np.empty((len(SERVE_OUT), n)), np.empty(n, dtype=np.int64)
    loop.wait(loop.submit(inp, p.mult, out, mult))
    for i, k in enumerate(SERVE_OUT):
        assert np.array_equal(out[i], plain[k]), k
    newton = loop.close()["newton"]
    assert [newton[k] for k in COUNTERS] == [c[k] for k in COUNTERS]
    s.close()
