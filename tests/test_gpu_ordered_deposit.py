"""Deterministic deposit on ragged patches against the oracle, bit for bit.

The kernel gives every 4^3-point tile of a patch's ghosted J a workgroup that
walks the clusters reaching it: the shapes have one, two and three clusters
per axis and patch (tiles that end inside and beyond the arrays), fast
particles (most change node), an empty species, one with particles in one
cell only (more than one batch of one tile) and one spread thinly.
"""
import numpy as np
import pytest

import smilei_amd as sa
from oracle import pyoracle as O
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,shape,patch", [(2, (8, 16, 24), (8, 8, 12)), (2, (12, 8, 20), (12, 8, 20)),
                                               (4, (12, 24, 16), (12, 12, 16)), (4, (20, 12, 12), (20, 12, 12))])
def test_ragged_patches_match_the_oracle(order, shape, patch):
    dx = (0.2, 0.25, 0.3)
    dt = cfl_dt(dx)
    g = sa.Simulation("3Dcartesian", order, shape, patch, dx, dt, deposit=sa.DEPOSIT_DETERMINISTIC)
    o = O.OracleSim(3, order, shape, patch, dx, dt)
    crowd = thermal(shape, dx, 1, 1.0, 3)
    n = len(crowd["x"])
    rng = np.random.default_rng(4)
    for d, k in enumerate("xyz"):
        crowd[k] = (shape[d] - 1 + rng.random(n)) * dx[d] * (1 - 1e-15)
    thin = {k: v[::29] for k, v in thermal(shape, dx, 1, 2.0, 5).items()}
    empty = {k: v[:0] for k, v in thin.items()}
    for q, p in ((-1.0, thermal(shape, dx, 3, 0.8, 1)), (2.0, empty), (-1.0, crowd), (1.0, thin)):
        load(g, g.add_species("s", 1.0, q, len(p["x"])), p)
        o.set_particles(o.add_species(1.0, q), *[p[k] for k in ("x", "y", "z", "px", "py", "pz", "w")])
    g.step(3)
    o.step(3)
    g.synchronize()
    for f in sa.FIELDS:
        assert np.array_equal(g.get_field(f), o.get_field(f)), f
