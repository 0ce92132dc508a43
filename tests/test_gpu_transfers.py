"""Droplets and records in and out of the device: every column and record word
at sizes around the tiles of the kernels (64 records, 256 droplets) and of the
staging buffer (128 MB: 381300 records, 493447 droplets at 34 columns), before
and after the slots have been reordered."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import COLUMNS, MODE_RK3, NREAL, PREC_FP64, Consts, DropletStep, Flags, Grid, Particles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    g = Grid.uniform(12, 10, 8, 0.02, 0.02, 0.02)
    s = DropletStep(g, Consts(dt=1e-7), Flags())
    shape = (12, 10, 10)
    s.set_fields(np.zeros(shape), np.zeros(shape), np.zeros(shape), np.full(shape, 300.0), np.full(shape, 0.02))
    yield s
    s.close()


def droplets(s, n):
    rng = np.random.default_rng(n)
    p = Particles.empty(n)
    p.soa[:] = rng.standard_normal((NREAL, n))
    g = s.grid
    p["x"], p["y"], p["z"] = rng.uniform(0, g.xl, n), rng.uniform(0, g.yl, n), rng.uniform(1e-4, g.zl - 1e-4, n)
    p["vx"] = p["vy"] = p["vz"] = 0.0
    p["radius"], p["Tp"], p["m_s"], p["kappa_s"] = 2e-5, 300.0, 1e-18, 1.2
    p.mult[:] = rng.integers(1, 1 << 40, n)
    p.pidx[:] = rng.integers(-(1 << 31), 1 << 31, n)
    p.procidx[:] = rng.integers(-(1 << 31), 1 << 31, n)
    return p


SIZES = [1, 63, 64, 65, 255, 257, 5000, 381_299, 381_301, 493_446, 493_449, 1_100_000]


@pytest.mark.parametrize("n", SIZES)
def test_round_trips(ctx, n):
    s, p = ctx, droplets(ctx, n)
    s.put(p)
    q = s.get()
    assert np.array_equal(q.soa, p.soa) and np.array_equal(q.mult, p.mult)
    assert np.array_equal(q.pidx, p.pidx) and np.array_equal(q.procidx, p.procidx)
    rec = s.get_records().view(np.float64).reshape(n, 44)
    ints = rec[:, :2].copy().view(np.int32)
    assert np.array_equal(ints[:, 0], p.pidx) and np.array_equal(ints[:, 1], p.procidx) and np.all(ints[:, 2:] == -1)
    assert np.array_equal(rec[:, 41].copy().view(np.int64), p.mult)
    assert np.array_equal(rec[:, 2:5].T, p.soa[[COLUMNS.index(c) for c in ("vx", "vy", "vz")]])
    raw = s.get_records().copy()
    s.put_records(raw)
    q = s.get()
    assert np.array_equal(q.soa, p.soa) and np.array_equal(q.mult, p.mult)
    assert np.array_equal(q.pidx, p.pidx) and np.array_equal(q.procidx, p.procidx)
    s.step(MODE_RK3, PREC_FP64, nsteps=1, it0=2)  # reorders the slots
    q = s.get()
    r = s.get_records().view(np.float64).reshape(n, 44)
    for w, c in ((5, "x"), (8, "ufx"), (17, "Tp"), (21, "radius"), (27, "m_s"), (40, "radiusold")):
        assert np.array_equal(r[:, w], q[c]), c
    assert np.array_equal(r[:, 41].copy().view(np.int64), p.mult) and np.array_equal(q.mult, p.mult)
    assert np.array_equal(r[:, :2].copy().view(np.int32)[:, 0], p.pidx)
    for c in ("x", "Tp", "ufz"):
        assert np.array_equal(s.column(c), q[c])


@pytest.mark.parametrize("mb", [0.9, 1.0, 1.1, 2.0, 3.99, 4.0, 16.0, 16.01, 33.3])
def test_large_fields_and_sources_pageable(mb):
    """Copies below, at and above the sizes at which they go through the pinned slots (1 MB) and wrap round them
    (4 x 4 MB): fields in by both layouts and sources out give the same bits."""
    nz = 30
    nx = 16
    ny = max(2, int(round(mb * 1e6 / 8 / ((nz + 2) * nx))))
    g = Grid.uniform(nx, ny, nz, 0.02, 0.02, 0.02)
    rng = np.random.default_rng(ny)
    f = [rng.standard_normal((nx, ny, nz + 2)) for _ in range(3)] + [300 + rng.random((nx, ny, nz + 2)), 0.02 * rng.random((nx, ny, nz + 2))]
    n = int(mb * 1e6 / 8)
    out = []
    for xp in (False, True):
        s = DropletStep(g, Consts(dt=1e-6), Flags())
        if xp:
            x = [np.zeros((nz + 2, ny, nx + 2)) for _ in f]
            for a, b in zip(x, f):
                a[:, :, :nx] = b.transpose(2, 1, 0)
            s.set_fields(*x, layout=2)
        else:
            s.set_fields(*f)
        s.put(droplets(s, n))
        s.interp(set_vp=True, set_tp=True)
        s.step(MODE_RK3, PREC_FP64, nsteps=1, it0=2)
        src = s.sources()
        ex = s.particle_coupling_exchange()
        out.append((s.get().soa, src, ex))
        s.close()
    (a, sa, ea), (b, sb, eb) = out
    assert np.array_equal(a, b)
    for u, v in zip((sa, *ea), (sb, *eb)):  # sums in an order that varies
        assert np.all(np.isfinite(u)) and np.max(np.abs(u - v)) <= 1e-12 * np.max(np.abs(u))
