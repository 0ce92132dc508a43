"""Ensembles drawn in put order (few droplets on a large grid) and in cell order (a
few more of them): the droplets that both hold have the same bits, as drawn, after
fused steps, after RK3 stages and in the records, from one ensemble and from three,
with both gathers."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import COLUMNS, MODE_BE, PREC_FP64, PREC_MIXED, Consts, DropletStep, Ensemble, Flags, Grid

pytestmark = pytest.mark.gpu

DIMS = (256, 256, 260)  # 257 x 257 x 261 cells: above 2^24, and 1024 x 16835 droplets
BELOW, ABOVE = 16_800, 16_900


@pytest.mark.parametrize("ilin", [1, 0])
@pytest.mark.parametrize("split", [None, (1, 5000)])
def test_same_droplets_in_both_orders(ilin, split):
    grid = Grid.uniform(*DIMS, 0.02, 0.02, 0.02)
    s = DropletStep(grid, Consts(dt=1e-5, radius_init=5e-6), Flags(ilin=ilin))
    rng = np.random.default_rng(17)
    base = rng.standard_normal((DIMS[0], DIMS[1], DIMS[2] + 2))
    s.set_fields(0.01 * base, 0.02 * base, -0.01 * base, 300 + 0.1 * base, 0.0225 + 1e-4 * base)

    def drawn(n):
        if split is None:
            s.generate(Ensemble(seed=5, first=7), n)
        else:
            s.generate([Ensemble(seed=5), Ensemble(seed=6, mult=3, kappa_s=0.6), Ensemble(seed=7)],
                       [split[0], split[1], n - sum(split)])

    def fused():
        s.step(MODE_BE, PREC_MIXED, nsteps=2, it0=2)
        s.step(MODE_BE, PREC_FP64, nsteps=1, it0=4)

    def stages():
        for it in (2, 3):
            for k in (1, 2, 3):
                s.particle_update_rk3(k, it=it, precision=PREC_FP64)
            s.particle_coupling_update(out=False)

    for then in (lambda: None, fused, stages):
        out = []
        for n in (BELOW, ABOVE):
            drawn(n)
            then()
            x = s.column("x")
            rec = s.get_records().reshape(n, 352)
            q = s.get()
            assert np.array_equal(x, q["x"])
            out.append((q, rec))
        (a, ra), (b, rb) = out
        for c in COLUMNS:
            assert np.array_equal(a[c], b[c][:BELOW]), c
        assert np.array_equal(a.pidx, b.pidx[:BELOW]) and np.array_equal(a.mult, b.mult[:BELOW])
        assert np.array_equal(ra, rb[:BELOW])
    s.close()
