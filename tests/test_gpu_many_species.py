"""Energies of more species than the reduction scratch is made for at first,
asked for as they are added, against sums over the loaded arrays."""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt, load, thermal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [sa.PLAIN_FP64, sa.MIXED])
def test_energies_of_many_species(form):
    shape, dx = (16, 16, 16), (0.2, 0.2, 0.2)
    sim = sa.Simulation("3Dcartesian", 2, shape, (8, 8, 8), dx, cfl_dt(dx), precision=form)
    want = []
    for s in range(11):
        p = thermal(shape, dx, 1, 0.2, s)
        load(sim, sim.add_species("s%d" % s, 1.0 + s, -1.0, len(p["x"])), p)
        want.append((1.0 + s) * np.sum(p["w"] * (np.sqrt(1 + p["px"] ** 2 + p["py"] ** 2 + p["pz"] ** 2) - 1)))
        got = sim.energies()
        assert len(got) == s + 2 and got[0] == 0.0
        np.testing.assert_allclose(got[1:], want, rtol=1e-11 if form == sa.PLAIN_FP64 else 1e-6, atol=0)
