"""Per-call updates of populations whose slots are put into cell order (8192
droplets and more) and of smaller ones, which stay in put order: 18 steps of
three particle_update_rk3 calls (past the 16th, where the slots are reordered),
with reads, an interpolation query and a coupling update between the calls,
give the bits of the fused steps in every column, and the coupling sources of
the fixed-order sum."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import COLUMNS, MODE_BE, MODE_RK3, PREC_FP64, PREC_MIXED, Consts, DropletStep, Flags, synth

from .helpers import mixed_droplets, small_grid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[1, 0], ids=["linear", "sixth"])
def start(request):
    rng = np.random.default_rng(5)
    grid, consts = small_grid("stretched"), Consts(dt=1e-6, radius_init=5e-6)
    s = DropletStep(grid, consts, Flags(ilin=request.param))
    s.set_fields(*synth.make_fields(grid, consts, rng, T0=300.0, T_sd=0.1, rh_uniform=(99, 101)))
    yield s, mixed_droplets(grid, rng, 20_000)
    s.close()


def set_up(s, p, n):
    q = type(p)(p.soa[:, :n].copy(), p.mult[:n].copy(), p.pidx[:n].copy(), p.procidx[:n].copy())
    s.put(q)
    s.interp(set_vp=True, set_tp=True)
    s.crit_radius()


@pytest.mark.parametrize("n", [64, 8191, 8192, 20_000])
@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
def test_rk3_calls_equal_fused_steps(start, n, prec):
    s, p = start
    set_up(s, p, n)
    s.step(MODE_RK3, prec, nsteps=18, it0=2)
    want = s.get()
    set_up(s, p, n)
    for it in range(2, 20):
        for stage in (1, 2, 3):
            s.particle_update_rk3(stage, it=it, precision=prec)
            if it == 5:
                s.column("xrhsx" if stage < 3 else "x")  # a read in the middle of a step
        if it % 7 == 0:
            box = s.particle_coupling_update()
            fixed = s.particle_coupling_update(deterministic=1)
            for a, b in zip(box, fixed):  # sums of at most n rounded terms, in two orders
                assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b)) + 1e-300
    got = s.get()
    for c in COLUMNS:
        assert np.array_equal(got[c], want[c]), c
    assert np.array_equal(got.pidx, want.pidx) and np.array_equal(got.mult, want.mult)


@pytest.mark.parametrize("n", [64, 8192, 20_000])
def test_statistics_and_queries_between_updates(start, n):
    """Statistics, the interpolation query and BE steps see the same droplets whether the record columns wait in slot
    order (after an update) or have been put into put order (after a read)."""
    s, p = start
    out = []
    for read in (False, True):
        set_up(s, p, n)
        for it in range(2, 6):
            for stage in (1, 2, 3):
                s.particle_update_rk3(stage, it=it, precision=PREC_FP64)
                if read:
                    s.get()
        s0, s1, lwp = s.particle_xy_stats()
        s.interp()
        s.step(MODE_BE, PREC_FP64, nsteps=1, it0=6)
        out.append((s0, s1, lwp, s.get()))
    (a0, a1, al, ap), (b0, b1, bl, bp) = out
    assert np.array_equal(a0[:3], b0[:3]) and np.array_equal(a0[9:], b0[9:]) and np.array_equal(a1[0], b1[0])
    for a, b in ((a0, b0), (a1, b1), (al, bl)):  # sums of n terms, in an order that varies
        assert np.all(np.abs(a - b) <= 1e-12 * np.max(np.abs(b), axis=-1, keepdims=True))
    for c in COLUMNS:
        assert np.array_equal(ap[c], bp[c]), c
