"""Canonical order inside crowded cells, against the oracle's, bit for bit.

The in-cell pass ranks cells of up to 256 particles with one lane per particle,
whole cells into batches of 512 places, and the rest by a workgroup: cells at
and around powers of two and every edge of these ranges appears as a cell's
number of particles, after one step in which a third of the particles change
cell (the fields are zero, so positions are the oracle's in every mode), for
several species of different sizes sorted in shared launches.
"""
import numpy as np
import pytest

import smilei_amd as sa
from oracle import pyoracle as O
from tests.plasma import cfl_dt, load

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 520]


def species(shape, dx, counts, seed):
    rng = np.random.default_rng(seed)
    nd = len(shape)
    pick = rng.choice(int(np.prod(shape)), len(counts), replace=False)
    cells = rng.permutation(np.repeat(pick, counts))
    n = len(cells)
    idx = np.unravel_index(cells, shape)
    pos = [(idx[d] + rng.random(n)) * dx[d] for d in range(nd)] + [np.zeros(n)] * (3 - nd)
    u = rng.normal(0.0, 0.3, (3, n)) * (rng.random(n) < 0.3)
    return dict(x=pos[0], y=pos[1], z=pos[2], px=u[0], py=u[1], pz=u[2], w=rng.random(n))


@pytest.mark.parametrize("mode,layout", [("det", 0), ("atomic", 0), ("atomic", 1)])
@pytest.mark.parametrize("shape,patch", [((8, 16, 12), (8, 8, 12)), ((48, 40), (16, 8))])
def test_crowded_cells(mode, layout, shape, patch):
    nd = len(shape)
    dx = (0.2, 0.25, 0.3)[:nd]
    dt = cfl_dt(dx)
    g = sa.Simulation("%dDcartesian" % nd, 2, shape, patch, dx, dt,
                      deposit=sa.DEPOSIT_DETERMINISTIC if mode == "det" else sa.DEPOSIT_ATOMIC)
    if mode == "atomic":
        g.set_tuning(sa.TUNE_INTERLEAVE, layout)
    o = O.OracleSim(nd, 2, shape, patch, dx, dt)
    for k, counts in enumerate((COUNTS, [3], COUNTS[:9] * 3, [], [257, 300, 64])):
        p = species(shape, dx, counts, k) if counts else {q: np.zeros(0) for q in ("x", "y", "z", "px", "py", "pz", "w")}
        load(g, g.add_species("s", 1.0, -1.0, len(p["x"])), p)
        o.set_particles(o.add_species(1.0, -1.0), *[p[q] for q in ("x", "y", "z", "px", "py", "pz", "w")])
    for step in range(2):  # as loaded, and after a step
        for s in range(5):
            a, b = g.get_particles(s), o.get_particles(s)
            for q in ("patch", "key", "x", "y", "px", "w"):
                assert np.array_equal(a[q], b[q]), (step, s, q)
        g.step(1)
        o.step(1)
    g.synchronize()
