"""The launch shape of untouched knobs where the particles lie in a few of the
grid's clusters: the particle kernel takes at most a tenth longer than with the
shape set by hand (1.2 times and more when the shape went by the grid).  And the
fields after steps agree to the order of the J sums (1e-12 of the largest
value, the bound of the tuning tests), also where a second species, loaded
later, is spread over the grid and changes the layout of the first.
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu


def plasma(shape, region, ppc, tuning=(), order=2, form=sa.PLAIN_FP64, widespread=False):
    nd = len(shape)
    dx = (0.2, 0.25, 0.3)[:nd]
    rng = np.random.default_rng(3)
    m = int(np.prod(region)) * ppc
    x = [(8 + rng.random(m) * r) * d for r, d in zip(region, dx)] + [np.zeros(m)] * (3 - nd)
    u = [0.05 * rng.standard_normal(m) for _ in range(3)]
    sim = sa.Simulation("%dDcartesian" % nd, order, shape, (16,) * nd, dx, cfl_dt(dx), precision=form)
    for k, v in tuning:
        sim.set_tuning(k, v)
    for q in (-1.0, 1.0):
        sim.set_particles(sim.add_species("s", 1.0, q, m), *x, *u, np.full(m, 1e-6))
    if widespread:
        p = thermal(shape, dx, 1, 0.1, 5, density=1e-5)
        load(sim, sim.add_species("t", 1.0, 1.0, len(p["x"])), p)
    return sim


def kernel_ms(sim):
    sim.step(3)
    times = [sim.profile_step()["particles"] for _ in range(15)]
    sim.synchronize()
    return min(times)


@pytest.mark.parametrize("case", ["mixed order 4", "2D"])
def test_untouched_knobs_cost_no_more(case):
    if case == "2D":
        args, by_hand = ((256, 256), (64, 64), 300), [(sa.TUNE_THREADS, 256)]
        kw = {}
    else:
        args, by_hand = ((64, 64, 64), (12, 12, 12), 300), [(sa.TUNE_INTERLEAVE, 1), (sa.TUNE_TILE, 1)]
        kw = dict(order=4, form=sa.MIXED)
    times = [[kernel_ms(plasma(*args, tuning=t, **kw)) for t in ((), by_hand)] for _ in range(3)]
    untouched, hand = (min(t) for t in zip(*times))
    assert untouched <= 1.1 * hand


@pytest.mark.parametrize("widespread", [False, True])
def test_layout_follows_the_loaded_species(widespread):
    kw = dict(order=4, form=sa.MIXED, widespread=widespread)
    a = plasma((48, 48, 32), (8, 8, 8), 5, **kw)
    b = plasma((48, 48, 32), (8, 8, 8), 5, tuning=[(sa.TUNE_INTERLEAVE, 1), (sa.TUNE_TILE, 1)], **kw)
    for sim in (a, b):
        sim.step(5)
        sim.synchronize()
    for f in sa.FIELDS:
        w = b.get_field(f)
        assert np.abs(a.get_field(f) - w).max() <= 1e-12 * np.abs(w).max(), f
