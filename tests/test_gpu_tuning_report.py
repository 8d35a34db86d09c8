"""smi_get_tuning reports the launch shape in effect, and setting a knob to the
value it reports changes nothing, whatever the order.
"""
import itertools

import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu

KNOBS = (sa.TUNE_THREADS, sa.TUNE_INTERLEAVE, sa.TUNE_TILE)


def make(form, order, shape, patch, ppc):
    nd = len(shape)
    dx = (0.2, 0.25, 0.3)[:nd]
    sim = sa.Simulation("%dDcartesian" % nd, order, shape, patch, dx, cfl_dt(dx),
                        precision=sa.MIXED if form == "mixed" else sa.PLAIN_FP64,
                        deposit=sa.DEPOSIT_DETERMINISTIC if form == "det" else sa.DEPOSIT_ATOMIC)
    p = thermal(shape, dx, ppc, 0.1, 3)
    load(sim, sim.add_species("s", 1.0, -1.0, len(p["x"])), p)
    return sim


def report(sim):
    return tuple(sim.get_tuning(k) for k in KNOBS)


CASES = [("fp64", 2, (16, 16, 16), (16, 16, 16), 2, (512, 1, 1)), ("fp64", 4, (24, 24, 12), (12, 12, 12), 1, (256, 1, 1)),
         ("fp64", 2, (96, 128), (32, 16), 3, (128, 1, 1)), ("fp64", 2, (96, 128), (32, 16), 80, (256, 1, 1)),
         ("fp64", 2, (96, 128), (32, 16), 250, (512, 1, 1)), ("det", 2, (16, 16, 16), (16, 16, 16), 2, (512, 1, 1)),
         ("mixed", 2, (32, 32, 32), (16, 16, 16), 2, (512, 1, 1)), ("mixed", 2, (48, 32, 32), (16, 16, 16), 2, (256, 1, 1)),
         ("mixed", 4, (32, 32, 32), (16, 16, 16), 2, (256, 1, 1)), ("mixed", 4, (48, 48, 32), (16, 16, 16), 2, (256, 2, 0))]


@pytest.mark.parametrize("form,order,shape,patch,ppc,want", CASES)
def test_the_values_in_effect(form, order, shape, patch, ppc, want):
    for knobs in itertools.permutations(range(3)):
        sim = make(form, order, shape, patch, ppc)
        assert report(sim) == want
        for k in knobs:
            if KNOBS[k] == sa.TUNE_INTERLEAVE and form == "det":
                continue
            sim.set_tuning(KNOBS[k], want[k])
            assert report(sim) == want
        sim.step(1)
        sim.synchronize()


def test_other_values_and_forms():
    shape, patch = (48, 48, 32), (16, 16, 16)
    for knob in (sa.TUNE_INTERLEAVE, sa.TUNE_TILE):
        sim = make("mixed", 4, shape, patch, 2)
        sim.set_tuning(knob, 1)
        assert report(sim) == (256, 1, 1)
    sim = make("mixed", 4, shape, patch, 2)
    sim.set_tuning(sa.TUNE_PERSISTENT, 1)
    assert report(sim) == (256, 1, 1)
    sim.set_tuning(sa.TUNE_PERSISTENT, 0)
    assert report(sim) == (256, 2, 0)
    best = sim.autotune(1)
    assert report(sim) == (best["threads"], best["interleave"], best["tile"])
    sim = make("mixed", 2, (32, 32, 32), patch, 2)
    sim.set_tuning(sa.TUNE_NODE_ACC, 1)  # a form of 256 threads
    assert report(sim) == (256, 1, 1)
