"""Launch shapes taken from the geometry against explicitly chosen ones.

The untouched knobs give 512 threads to the smallest grids, 128 to 2D ones and
the pair-interleaved layout to the order-4 mixed form; only the order of the J
sums may differ from the starting values set by hand.  FP64: 11 steps from
equal states drift by rounding (1e-12 of the largest value, the bound of the
tuning tests); mixed: the tile sums are exact, so fields agree to the FP64
flush order, 1e-12 as well.
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,order,shape,patch,ppc", [
    ("fp64", 2, (24, 16, 16), (8, 8, 16), 5), ("fp64", 4, (24, 12, 12), (12, 12, 12), 3),
    ("fp64", 2, (16, 32), (16, 8), 9), ("fp64", 2, (96, 128), (32, 16), 3),
    ("mixed", 2, (32, 24, 16), (16, 8, 16), 5), ("mixed", 2, (32, 40, 32), (16, 8, 16), 3),
    ("mixed", 4, (24, 24, 12), (12, 24, 12), 3), ("mixed", 4, (36, 24, 48), (12, 24, 24), 2)])
def test_untouched_knobs(form, order, shape, patch, ppc):
    nd = len(shape)
    dx = (0.2, 0.25, 0.3)[:nd]
    sims = []
    for explicit in (False, True):
        sim = sa.Simulation("%dDcartesian" % nd, order, shape, patch, dx, cfl_dt(dx),
                            precision=sa.MIXED if form == "mixed" else sa.PLAIN_FP64)
        if explicit:
            for k in (sa.TUNE_INTERLEAVE, sa.TUNE_THREADS, sa.TUNE_TILE):
                sim.set_tuning(k, sim.get_tuning(k))
        for s, (m, q) in enumerate(((1.0, -1.0), (1836.0, 1.0))):
            p = thermal(shape, dx, ppc, 0.3 / np.sqrt(m), 3 + s)
            load(sim, sim.add_species("s", m, q, len(p["x"])), p)
        sim.step(10)
        sim.synchronize()
        sims.append(sim)
    for f in sa.FIELDS:
        a, b = (sim.get_field(f) for sim in sims)
        scale = np.abs(b).max()
        assert np.abs(a - b).max() <= 1e-12 * scale, f
    # switching a knob afterwards re-stores the state in the chosen layout
    sims[0].set_tuning(sa.TUNE_INTERLEAVE, 0)
    sims[0].step(1)
    sims[1].step(1)
    sims[0].synchronize()
    a, b = sims[0].rho(), sims[1].rho()
    assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
