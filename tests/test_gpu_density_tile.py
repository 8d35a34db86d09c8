"""Charge density of a resident simulation (smi_rho) against a direct sum.

The density kernels sum each 4^ND cluster's particles on a tile in LDS: the
cases put particles on the faces of clusters, patches and the periodic box
(nodes at both ends of the tile), leave clusters empty or with one particle,
and fill one cell with more particles than a workgroup has threads.

Every node is a sum of m <= (particles) products of FP64 weights; reordering
it moves it by at most m * 2^-53 * sum|terms|.  With the largest node holding
at most 600 * 2 contributions the bound is 1200 * 1.1e-16 < 2e-13 of the
largest |rho|.  The mixed form rounds offsets and weights to FP32 (2^-24
each, 3 factors of slope <= 2 per cell): 1e-6 of the largest value.
"""
import numpy as np
import pytest

import smilei_amd as sa
from tests.plasma import cfl_dt

pytestmark = pytest.mark.gpu


def spline(order, d):
    if order == 2:
        return np.stack([0.5 * (d - 0.5) ** 2, 0.75 - d * d, 0.5 * (d + 0.5) ** 2])
    return np.stack([(1 - 2 * d) ** 4 / 384, 19 / 96 - 11 * d / 24 + d ** 2 / 4 + d ** 3 / 6 - d ** 4 / 6,
                     115 / 192 - 5 * d ** 2 / 8 + d ** 4 / 4, 19 / 96 + 11 * d / 24 + d ** 2 / 4 - d ** 3 / 6 - d ** 4 / 6,
                     (1 + 2 * d) ** 4 / 384])


def direct(shape, dx, order, pos, cw):
    nd, H = len(dx), order // 2
    rho = np.zeros(shape[:nd])
    pn = [pos[d] / dx[d] for d in range(nd)]
    node = [np.floor(p + 0.5).astype(int) for p in pn]
    S = [spline(order, pn[d] - node[d]) for d in range(nd)]
    for off in np.ndindex(*([order + 1] * nd)):
        v = cw.copy()
        for d in range(nd):
            v = v * S[d][off[d]]
        np.add.at(rho, tuple((node[d] + off[d] - H) % shape[d] for d in range(nd)), v)
    return rho


def positions(shape, dx, seed):
    """Random particles, some at cluster / patch / box faces, one crowded cell."""
    rng = np.random.default_rng(seed)
    nd = len(dx)
    n = 257
    cells = np.stack([rng.integers(0, shape[d], n) for d in range(nd)])
    frac = rng.random((nd, n))
    faces = rng.random((nd, n)) < 0.3
    cells = np.where(faces, cells // 4 * 4, cells)
    frac = np.where(faces, rng.choice([0.0, 1e-12, 0.5, 1 - 1e-12], (nd, n)), frac)
    crowd = np.tile(np.array([[s - 1] for s in shape[:nd]]), (1, 600))
    cells = np.concatenate([cells, crowd], 1)
    frac = np.concatenate([frac, rng.random((nd, 600))], 1)
    pos = [np.minimum((cells[d] + frac[d]) * dx[d], np.nextafter(shape[d] * dx[d], 0.0)) for d in range(nd)]
    return pos, rng.random(n + 600) + 0.5


@pytest.mark.parametrize("form,order,shape,patch", [
    ("fp64", 2, (16, 8, 24), (8, 8, 12)), ("fp64", 4, (24, 12, 12), (12, 12, 12)), ("fp64", 2, (24, 16, 1), (8, 16, 1)),
    ("mixed", 2, (16, 8, 24), (8, 8, 12)), ("mixed", 4, (24, 12, 12), (12, 12, 12))])
@pytest.mark.parametrize("layout", [0, 1])
def test_density_tile(form, order, shape, patch, layout):
    nd = 2 if shape[2] == 1 else 3
    dx = (0.2, 0.25, 0.3)[:nd]
    sim = sa.Simulation("%dDcartesian" % nd, order, shape[:nd], patch[:nd], dx, cfl_dt(dx),
                        precision=sa.MIXED if form == "mixed" else sa.PLAIN_FP64)
    sim.set_tuning(sa.TUNE_INTERLEAVE, layout)
    pos, w = positions(shape, dx, 11)
    want = np.zeros(shape[:nd])
    for s, q in enumerate((-1.0, 3.0)):
        sid = sim.add_species("s%d" % s, 1.0, q, len(w))
        p = [v[s::2] for v in pos]
        z = p[2] if nd == 3 else np.zeros(len(w[s::2]))
        u = np.zeros(len(z))
        sim.set_particles(sid, p[0], p[1], z, u, u, u, w[s::2])
        want += direct(shape, dx, order, p, q * w[s::2] / np.prod(dx))
    got = sim.rho().reshape(shape[:nd])
    tol = 1e-6 if form == "mixed" else 2e-13
    assert np.abs(got - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("shape,patch", [((8, 8, 12), (8, 8, 12)), ((16, 8, 8), (8, 8, 8)), ((20, 12), (20, 12)),
                                         ((8, 16), (8, 8))])
def test_deterministic_density_is_the_ordered_sum(shape, patch):
    """The fixed-order density, bit for bit: per node, the cells that reach it
    in x, y, z order, their particles in sorted order, products ((cw Sx) Sy) Sz."""
    nd = len(shape)
    dx = (0.2, 0.25, 0.3)[:nd]
    sim = sa.Simulation("%dDcartesian" % nd, 2, shape, patch, dx, cfl_dt(dx), deposit=sa.DEPOSIT_DETERMINISTIC)
    pos, w = positions(shape + (1,) * (3 - nd), dx, 5)
    pos, w = [v[:400] for v in pos], w[:400]
    sid = sim.add_species("s", 1.0, -2.0, len(w))
    zero = np.zeros(len(w))
    sim.set_particles(sid, pos[0], pos[1], pos[2] if nd == 3 else zero, zero, zero, zero, w)
    p = sim.get_particles(sid)
    x = [p[k] for k in "xyz"[:nd]]
    dinv = [1.0 / v for v in dx]
    node = [np.floor(x[d] * dinv[d] + 0.5).astype(int) for d in range(nd)]
    cell = [np.minimum(np.floor(x[d] * dinv[d]).astype(int), shape[d] - 1) for d in range(nd)]
    S = []
    for d in range(nd):
        e = x[d] * dinv[d] - node[d]
        S.append([0.5 * (e * e - e + 0.25), 0.75 - e * e, 0.5 * (e * e + e + 0.25)])
    vol = 1.0
    for v in dx:
        vol *= v
    cw = (1.0 / vol * -2.0) * p["w"]
    by_cell = {}
    for i, c in enumerate(zip(*cell)):
        by_cell.setdefault(c, []).append(i)
    want = np.zeros(shape)
    for n in np.ndindex(*shape):
        acc = 0.0
        for off in np.ndindex(*([4] * nd)):
            cu = [n[d] - 2 + off[d] for d in range(nd)]
            for i in by_cell.get(tuple(cu[d] % shape[d] for d in range(nd)), ()):
                o = [n[d] - (node[d][i] + cu[d] - cu[d] % shape[d] - 1) for d in range(nd)]
                if all(0 <= v < 3 for v in o):
                    t = cw[i]
                    for d in range(nd):
                        t = t * S[d][o[d]][i]
                    acc += t
        want[n] = acc
    assert np.array_equal(sim.rho().reshape(shape), want)
