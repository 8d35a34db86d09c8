"""Momenta of the atomic FP64 form after one step in a uniform magnetic field
that turns them by more than a right angle: no further from extended precision
(rms over the particles) than those of the deterministic form, which gathers
and pushes in the reference's association.

|t| = |q dt B / 2 m gamma| is 5 to 1,000.
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [5.0, 50.0, 1000.0])
@pytest.mark.parametrize("nd,order", [(2, 2), (3, 2), (3, 4)])
def test_rounding_of_a_strong_rotation(nd, order, t):
    shape, patch = ((64, 48), (16, 24)) if nd == 2 else ((32, 16, 16), (16, 16, 16))
    dx = (0.2, 0.25, 0.3)[:nd]
    dt = cfl_dt(dx)
    p = thermal(shape, dx, 4 if nd == 3 else 10, 0.05, 7, density=1e-9)
    n = len(p["x"])
    p["w"] = p["w"] * (1.0 + np.arange(n) / n)  # tells the particles apart
    b = np.array([0.36, -0.48, 0.8]) * t / (0.5 * dt)
    u = np.stack([p[k][np.argsort(p["w"])] for k in ("px", "py", "pz")]).astype(np.longdouble)
    tv = (-0.5 * np.longdouble(dt) / np.sqrt(1 + (u * u).sum(0))) * b.astype(np.longdouble)[:, None]
    s = 2 * tv / (1 + (tv * tv).sum(0))
    want = u + np.cross(u + np.cross(u, tv, axis=0), s, axis=0)
    rms = []
    for deposit in (sa.DEPOSIT_ATOMIC, sa.DEPOSIT_DETERMINISTIC):
        sim = sa.Simulation("%dDcartesian" % nd, order, shape, patch, dx, dt, deposit=deposit)
        load(sim, sim.add_species("s", 1.0, -1.0, n), p)
        for k, v in zip("xyz", b):
            for f in ("B" + k, "B%s_m" % k):
                sim.set_field(f, np.full(sim.get_field(f).shape, v))
        sim.step(1)
        q = sim.get_particles(0)
        sim.synchronize()
        got = np.stack([q[k][np.argsort(q["w"])] for k in ("px", "py", "pz")])
        rms.append(float(np.sqrt((((got - want) ** 2).sum(0) / (want * want).sum(0)).mean())))
    assert rms[0] <= rms[1]
