"""Per-call steps after a put, on both sides of the lines from which the first one
puts the slots into cell order (32768 droplets, a 32nd of the cells, a coupling
flag), from which the second one does, and of a sparse grid, on which none does:
three steps of three stages with the coupling update between them give the bits of
the fused steps in every column, and each droplet those of a smaller population."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import COLUMNS, MODE_RK3, PREC_FP64, Consts, DropletStep, Flags, Grid, Particles, synth

from .helpers import mixed_droplets

pytestmark = pytest.mark.gpu

DENSE, WIDE = (20, 16, 30), (128, 96, 96)  # 32 x 32768 droplets are fewer than WIDE's cells


@pytest.mark.parametrize("dims,n", [(DENSE, 32_767), (DENSE, 32_768), (WIDE, 32_768), (WIDE, 40_000), (WIDE, 8_192)])
@pytest.mark.parametrize("coupled", [1, 0])
def test_steps_after_a_put(dims, n, coupled):
    rng = np.random.default_rng(n)
    grid, consts = Grid.uniform(*dims, 0.02, 0.025, 0.03), Consts(dt=1e-6, radius_init=5e-6)
    s = DropletStep(grid, consts, Flags(icouple=coupled, iTcouple=coupled, iHcouple=coupled))
    s.set_fields(*synth.make_fields(grid, consts, rng, T0=300.0, T_sd=0.1, rh_uniform=(99, 101)))
    p = mixed_droplets(grid, rng, n)
    p["Tp"] = 300.0
    out = []
    for way, m in (("fused", n), ("calls", n), ("calls after interp", n), ("calls", 500)):
        s.put(Particles(p.soa[:, :m].copy(), p.mult[:m].copy(), p.pidx[:m].copy(), p.procidx[:m].copy()))
        if way.endswith("interp"):
            s.interp(set_vp=True, set_tp=True)
            s.put(p)  # what follows it is a first pass again
        if way == "fused":
            s.step(MODE_RK3, PREC_FP64, nsteps=3, it0=2)
        else:
            for it in (2, 3, 4):
                for stage in (1, 2, 3):
                    s.particle_update_rk3(stage, it=it, precision=PREC_FP64)
                if coupled:
                    s.particle_coupling_update(out=False)
        out.append(s.get())
    s.close()
    for q in out[1:]:
        for c in COLUMNS:
            assert np.array_equal(q[c], out[0][c][: q.n]), c
        assert np.array_equal(q.pidx, out[0].pidx[: q.n]) and np.array_equal(q.mult, out[0].mult[: q.n])
