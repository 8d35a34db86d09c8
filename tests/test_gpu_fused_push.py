"""Fused gather and push of the atomic FP64 form against the reference-order ones
of the deterministic form, one step from the same state.

Weak and strong fields, thermal and ultra-relativistic momenta.  A gathered
component sums at most 125 products (both forms round each a few times, so
260 eps of the largest |field| bounds the difference); the push adds a few tens
of eps of the momentum, and an error of t = q dt B / 2m turns the momentum by
twice that.  The position follows with dt.
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


@pytest.mark.parametrize("field,sigma", [(0.01, 0.05), (50.0, 0.05), (0.01, 1000.0), (50.0, 1000.0)])
@pytest.mark.parametrize("nd,order", [(2, 2), (3, 2), (3, 4)])
def test_one_step(nd, order, field, sigma):
    shape, patch = ((32, 24), (16, 8)) if nd == 2 else ((32, 16, 16), (16, 16, 16))
    dx = (0.2, 0.25, 0.3)[:nd]
    dt = cfl_dt(dx)
    p = thermal(shape, dx, 6, sigma, 7, density=1e-9)
    n = len(p["x"])
    p["w"] = p["w"] * (1.0 + np.arange(n) / n)  # tells the particles apart
    rng = np.random.default_rng(3)
    names = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")
    got = []
    for deposit in (sa.DEPOSIT_ATOMIC, sa.DEPOSIT_DETERMINISTIC):
        sim = sa.Simulation("%dDcartesian" % nd, order, shape, patch, dx, dt, deposit=deposit)
        load(sim, sim.add_species("s", 1.0, -1.0, n), p)
        rng = np.random.default_rng(3)
        for k in names:
            f = field * rng.uniform(-1.0, 1.0, sim.get_field(k).shape)
            sim.set_field(k, f)
            if k[0] == "B":
                sim.set_field(k + "_m", f)
        sim.step(1)
        q = sim.get_particles(0)
        o = np.argsort(q["w"])
        got.append({k: np.asarray(q[k])[o] for k in ("x", "y", "z", "px", "py", "pz", "w")})
        sim.synchronize()
    a, b = got
    assert np.array_equal(a["w"], b["w"])
    umax = max(np.abs(b[k]).max() for k in ("px", "py", "pz"))
    t = 0.5 * dt * field
    tol = EPS * (100.0 * umax + 2 * 520.0 * t * umax + 2 * 260.0 * t)
    for k in ("px", "py", "pz"):
        assert np.abs(a[k] - b[k]).max() <= tol
    assert umax > 0.1 * min(1.0, field * dt)
    for d, k in enumerate("xyz"[:nd]):
        length = shape[d] * dx[d]
        diff = np.abs(a[k] - b[k])
        assert np.minimum(diff, length - diff).max() <= dt * tol + 4 * EPS * length
