"""Momenta whose square overflows: gamma is infinite and 1/gamma zero, so the
particle keeps its momentum and its place, in the atomic FP64 form as in the
deterministic one, and the particles beside it move as without it.
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd,order", [(2, 2), (3, 2), (3, 4)])
def test_squares_that_overflow(nd, order):
    shape, patch = ((16, 16), (16, 16)) if nd == 2 else ((16, 16, 16), (16, 16, 16))
    dx = (0.2, 0.25, 0.3)[:nd]
    dt = cfl_dt(dx)
    p = thermal(shape, dx, 1, 0.05, 7, density=1e-9)
    n = len(p["x"])
    p["w"] = p["w"] * (1.0 + np.arange(n) / n)  # tells the particles apart
    for k, v in zip(("px", "py", "pz"), (2e160, -1e155, 1e200)):
        p[k][::17] = v
    out = []
    for deposit in (sa.DEPOSIT_ATOMIC, sa.DEPOSIT_DETERMINISTIC):
        sim = sa.Simulation("%dDcartesian" % nd, order, shape, patch, dx, dt, deposit=deposit)
        load(sim, sim.add_species("s", 1.0, -1.0, n), p)
        for f in ("Bx", "Bx_m", "Bz", "Bz_m"):
            sim.set_field(f, np.full(sim.get_field(f).shape, 0.5))
        sim.step(1)
        sim.synchronize()
        q = sim.get_particles(0)
        o = np.argsort(q["w"])
        out.append({k: q[k][o] for k in ("x", "y", "z", "px", "py", "pz")})
        assert all(np.isfinite(sim.get_field(f)).all() for f in sa.FIELDS)
    a, b = out
    for k in ("x", "y", "z")[:nd] + ("px", "py", "pz"):
        assert np.array_equal(a[k][::17], p[k][np.argsort(p["w"])][::17]), k
        assert np.array_equal(a[k][::17], b[k][::17]), k
        scale = np.abs(b[k][np.arange(n) % 17 != 0]).max()
        assert np.abs(a[k] - b[k])[np.arange(n) % 17 != 0].max() <= 1e-13 * scale, k
