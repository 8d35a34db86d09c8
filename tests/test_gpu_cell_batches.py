"""Canonical order inside cells where a wavefront takes 16, 32 or 64 cells.

The in-cell pass gives a wavefront 64 cells on grids of 5.2e5 cells (of all
species) and more, 32 from 2.6e5 on, 16 below, and ranks as many whole cells
at a time as fit into 512 places.  The run of cells here makes batches that
end exactly at 512 places, one place short of it and with a cell that no
longer fits, next to empty cells, single particles and cells beyond 256, which
another kernel takes.  Order and destinations are whole numbers: equal to the
oracle's, as loaded and after a step in which a third of the particles move.
"""
import numpy as np
import pytest

import smilei_amd as sa
from oracle import pyoracle as O
from tests.plasma import cfl_dt, load

pytestmark = pytest.mark.gpu

RUN = [256, 256, 1, 0, 255, 256, 2, 0, 0, 511 - 257, 3, 257, 200, 200, 111, 1, 64, 64, 0, 7, 256, 300, 1] + [8] * 41 + [33] * 64


def species(shape, dx, nspread, seed):
    """RUN on consecutive cells at both ends and in the middle, the rest thin."""
    rng = np.random.default_rng(seed)
    ncell = int(np.prod(shape))
    cells = [rng.integers(0, ncell, nspread)]
    for start in (0, ncell // 2 - 5, ncell - len(RUN)):
        cells.append(np.repeat(np.arange(start, start + len(RUN)), RUN))
    cells = rng.permutation(np.concatenate(cells))
    idx = np.unravel_index(cells, shape)
    n = len(cells)
    pos = [(idx[d] + rng.random(n)) * dx[d] for d in range(2)]
    u = rng.normal(0.0, 0.3, (3, n)) * (rng.random(n) < 0.3)
    return dict(x=pos[0], y=pos[1], z=np.zeros(n), px=u[0], py=u[1], pz=u[2], w=rng.random(n))


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("shape", [(256, 128), (512, 512), (1024, 512)])
def test_batches_of_cells(shape, layout):
    dx = (0.2, 0.25)
    dt = cfl_dt(dx)
    g = sa.Simulation("2Dcartesian", 2, shape, (64, 32), dx, dt)
    g.set_tuning(sa.TUNE_INTERLEAVE, layout)
    o = O.OracleSim(2, 2, shape, (64, 32), dx, dt)
    p = species(shape, dx, 40000, 3)
    load(g, g.add_species("s", 1.0, -1.0, len(p["x"])), p)
    o.set_particles(o.add_species(1.0, -1.0), *[p[q] for q in ("x", "y", "z", "px", "py", "pz", "w")])
    for step in range(2):
        a, b = g.get_particles(0), o.get_particles(0)
        for q in ("patch", "key", "x", "y", "px", "w"):
            assert np.array_equal(a[q], b[q]), (step, q)
        g.step(1)
        o.step(1)
    g.synchronize()
