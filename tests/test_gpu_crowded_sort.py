"""The sort's time where the crowded cells lie together: 16^3 cells of 130 or 300
particles in a grid of 64^3 are sorted in less than three times the time of
the same number of particles spread over twice as many cells per axis (about
twice; 14 and 5 times when a wavefront worked on its run of 64 crowded cells
alone, and few workgroups on the most crowded ones).
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt

pytestmark = pytest.mark.gpu

DX = (0.2, 0.25, 0.3)


def sort_ms(width, ppc):
    rng = np.random.default_rng(3)
    m = width ** 3 * ppc
    x = [(16 + rng.random(m) * width) * DX[d] for d in range(3)]
    u = [0.05 * rng.standard_normal(m) for _ in range(3)]
    sim = sa.Simulation("3Dcartesian", 2, (64, 64, 64), (16, 16, 16), DX, cfl_dt(DX))
    for q in (-1.0, 1.0):
        sim.set_particles(sim.add_species("s", 1.0, q, m), *x, *u, np.full(m, 1e-6))
    sim.step(3)
    times = [sim.profile_step()["sort"] for _ in range(15)]
    sim.synchronize()
    return min(times)


@pytest.mark.parametrize("ppc", [136, 296])
def test_crowded_cells_side_by_side(ppc):
    assert sort_ms(16, ppc) <= 3 * sort_ms(32, ppc // 8)
