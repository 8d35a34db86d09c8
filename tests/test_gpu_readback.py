"""Fields read back through each staging path, byte for byte.

Below, at and above the size where the path changes (4 MiB), with
whole and ragged last blocks, several fields in a row (the staging is reused)
and with steps still running on the context's stream; energies of several
species against sums over the returned arrays.
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu

DX = (0.2, 0.2, 0.2)


@pytest.mark.parametrize("shape", [(8, 8, 8), (128, 32, 32), (136, 32, 32), (120, 64, 64), (128, 64, 64), (136, 64, 64),
                                   (1024, 64, 24)])
def test_fields_come_back_as_set(shape):
    sim = sa.Simulation("3Dcartesian", 2, shape, (8, 8, 8), DX, cfl_dt(DX))
    rng = np.random.default_rng(1)
    want = {f: rng.random(shape) for f in sa.FIELDS[:4]}
    for f, a in want.items():
        sim.set_field(f, a)
    for _ in range(2):
        for f, a in want.items():
            assert np.array_equal(sim.get_field(f), a), f


def test_read_back_waits_for_the_steps():
    shape = (128, 64, 72)
    sims = [sa.Simulation("3Dcartesian", 2, shape, (16, 16, 24), DX, cfl_dt(DX)) for _ in range(2)]
    rng = np.random.default_rng(2)
    e = {f: rng.random(shape) for f in ("Ex", "Ey", "Bz")}
    for sim in sims:
        for f, a in e.items():
            sim.set_field(f, a)
    sims[0].step(30)
    sims[1].step(30)
    sims[1].synchronize()
    for f in sa.FIELDS:
        assert np.array_equal(sims[0].get_field(f), sims[1].get_field(f)), f


def test_energies_of_several_species():
    shape = (16, 16, 16)
    sim = sa.Simulation("3Dcartesian", 2, shape, (8, 8, 8), DX, cfl_dt(DX))
    want = []
    for s, (m, n) in enumerate(((1.0, 3), (1836.0, 1), (2.0, 0), (4.0, 5))):
        p = {k: v[:len(v) * min(n, 1)] for k, v in thermal(shape, DX, max(n, 1), 0.2, s).items()}
        load(sim, sim.add_species("s", m, -1.0, len(p["x"])), p)
        g = np.sqrt(1 + p["px"] ** 2 + p["py"] ** 2 + p["pz"] ** 2)
        want.append(m * np.sum(p["w"] * (g - 1)))
    got = sim.energies()
    assert got[0] == 0.0
    np.testing.assert_allclose(got[1:], want, rtol=1e-11, atol=0)
