"""The cell statistics where cells hold many droplets: by an atomic for each droplet
(after a put) and by runs of the cell sort; every number of lanes that a cell's
run is shared by (1 to 64, by the mean number of droplets in a cell), with and
without a cluster in one cell whose run the whole wave shares, in columns at the
edge of the box and inside, against the oracle.  Counts are exact; sums of n
positive terms in two orders differ by 2 n eps at most."""
from __future__ import annotations

import numpy as np
import pytest

from ntlp_amd import Consts, DropletStep, Flags
from ntlp_amd.grid import Grid
from oracle import Oracle

from .helpers import mixed_droplets

pytestmark = pytest.mark.gpu

MEANS = [0.5, 3.1, 6.1, 12.5, 25.0, 49.0, 97.0, 400.0]  # 1, 2, 4, 8, 16, 32, 64 and 64 lanes


@pytest.mark.parametrize("mean", MEANS)
@pytest.mark.parametrize("cluster", [None, (0, 0, 0), (4, 3, 2), (6, 4, 12)])
def test_counts_and_tauc(mean, cluster):
    grid, consts = Grid.tanh_stretched(7, 5, 13, 0.02, 0.025, 0.005, 0.03), Consts(radius_init=5e-6)
    rng = np.random.default_rng(int(10 * mean))
    n = int(round(mean * grid.nnx * grid.nny * grid.nnz))
    p = mixed_droplets(grid, rng, n)
    for d, top in (("x", grid.xl), ("y", grid.yl), ("z", grid.zl)):
        p[d] = rng.uniform(-0.01, 1.01, n) * top
    if cluster is not None:
        i, j, k = cluster
        m = np.flatnonzero(rng.random(n) < 0.4)
        p["x"][m], p["y"][m] = (i + rng.random(m.size)) * grid.dx, (j + rng.random(m.size)) * grid.dy
        p["z"][m] = grid.z[k] + rng.random(m.size) * (grid.z[k + 1] - grid.z[k])
    p.mult[:] = rng.integers(1, 2000, n)
    ora = Oracle(grid, consts, Flags())
    s = DropletStep(grid, consts, Flags())
    s.set_fields(*[np.zeros((grid.nnx, grid.nny, grid.nnz + 2))] * 5)  # present, not read
    s.put(p)
    counts, tauc = ora.wcell_counts(p["x"], p["y"], p["z"]), ora.calc_tauc_min(p.soa, p.mult)
    for by_runs in (False, True):
        if by_runs:  # the coupling update leaves the sort
            s.particle_coupling_update(out=False)
        assert np.array_equal(s.wcell_counts(), counts), by_runs
        assert abs(s.calc_tauc_min() / tauc - 1) < 4.5e-16 * n + 1e-13, by_runs
    s.close()


def test_a_cluster_takes_no_longer_than_its_droplets():
    """A tenth of a million droplets in one cell: the queries stay within sixty
    times those of the same number spread evenly (25; one lane for the run: 800)."""
    grid = Grid.uniform(128, 128, 128, 0.02, 0.02, 0.02)
    s = DropletStep(grid, Consts(radius_init=5e-6), Flags())
    s.set_fields(*[np.zeros((128, 128, 130))] * 5)
    rng = np.random.default_rng(5)
    took = []
    for some in (0, 100_000):
        p = mixed_droplets(grid, rng, 1_000_000)
        p["x"][:some], p["y"][:some], p["z"][:some] = (40.5 * d for d in (grid.dx, grid.dy, 0.02))
        s.put(p)
        s.particle_coupling_update(out=False)  # leaves the sort
        for timed in (False, True):
            s.timing(timed)
            s.wcell_counts()
            s.calc_tauc_min()
        took.append(sum(ms for name, (_, ms) in s.kernel_times().items() if name in ("wcells", "tauc")))
        s.timing(False)
    s.close()
    assert took[1] < 60 * took[0], took
