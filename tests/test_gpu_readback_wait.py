"""A field read while steps are still running: the host threads that copy it
out sleep until the first block is there.

The calling thread may spin on the stream (one second of processor time a
second); four helpers that spin too make it five.
"""
import time

import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu


def test_waiting_for_the_steps_takes_one_processor():
    shape, dx = (128, 64, 72), (0.2, 0.25, 0.3)
    sim = sa.Simulation("3Dcartesian", 2, shape, (16, 16, 24), dx, cfl_dt(dx))
    p = thermal(shape, dx, 4, 0.1, 3)
    load(sim, sim.add_species("s", 1.0, -1.0, len(p["x"])), p)
    sim.step(2)
    want = sim.get_field("Ex")  # warm
    sim.step(200)
    cpu, wall = time.process_time(), time.perf_counter()
    got = sim.get_field("Ex")
    cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    assert wall > 0.03
    assert cpu <= 2.5 * wall
    assert np.isfinite(got).all() and not np.array_equal(got, want)
