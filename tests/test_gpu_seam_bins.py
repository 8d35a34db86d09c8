"""Device projector seam on awkward bins against smi_currents_3d in index order
and smi_density_3d.

Bins that are empty, hold one particle, or more node changers than the
kernel's queue; both loop orders.  The sums are reordered and the weights
factorised: a point gets fewer than 3,000 contributions, so 3,000 * 2^-53 of
the largest |value| (4e-13) bounds the difference.
"""
import ctypes

import numpy as np
import pytest

from smilei_amd import _lib
from tests.plasma import cfl_dt

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DX = (0.2, 0.25, 0.3)
N = (8, 12, 8)


def p(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("cell_sorting", [False, True])
@pytest.mark.parametrize("crowd,moving", [(0, 0.1), (1, 0.5), (700, 1.0)])
def test_bins(cell_sorting, crowd, moving):
    rng = np.random.default_rng(crowd + 1)
    nb = [v // 4 for v in N]
    counts = rng.integers(0, 90, int(np.prod(nb)))
    counts[::5] = 0
    counts[3] = crowd
    m = int(counts.sum())
    b = np.repeat(np.arange(len(counts)), counts)
    bc = np.stack([b // (nb[1] * nb[2]), b // nb[2] % nb[1], b % nb[2]])
    pn = 4 * bc + 4 * rng.random((3, m))
    node = np.floor(pn + 0.5)
    new = pn + rng.uniform(-0.95, 0.95, (3, m)) * (rng.random(m) < moving)
    charge = rng.integers(-3, 4, m).astype(np.int16)
    w = rng.random(m) + 0.5
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    x = [dev(new[d] * DX[d]) for d in range(3)]
    iold, delta, dw, dq = dev((node + 2).astype(np.int32)), dev(pn - node), dev(w), dev(charge)
    ends, inv = dev(np.cumsum(counts).astype(np.int32)), dev(np.ones(m))
    shapes = [[N[d] + 5 + (d == c) for d in range(3)] for c in range(3)] + [[v + 5 for v in N]]
    got = [torch.zeros(s, dtype=torch.float64, device="cuda") for s in shapes]
    want = [torch.zeros(s, dtype=torch.float64, device="cuda") for s in shapes]
    dt, vol, L = cfl_dt(DX), float(np.prod(DX)), _lib.load()
    tail = ([p(t) for t in x] + [p(dq), p(dw), p(ends)] + nb + [p(inv), p(iold), p(delta), m, 1.0 / vol]
            + [1.0 / v for v in DX] + [v / dt for v in DX] + [-2, -2, -2, N[1] + 5, N[2] + 5, 1, cell_sorting])
    torch.cuda.synchronize()
    _lib.check(L.smi_current_deposition_3d(*[p(t) for t in got[:3]], *[t.numel() for t in got[:3]], *tail))
    _lib.check(L.smi_density_deposition_3d(p(got[3]), got[3].numel(), *tail))
    ints, size = (ctypes.c_int * 3)(-2, -2, -2), (ctypes.c_int * 3)(*[v + 5 for v in N])
    wq = dev(charge * w)
    _lib.check(L.smi_currents_3d(2, *[p(t) for t in want[:3]], size, ints, (ctypes.c_double * 3)(*DX), dt, 1.0, m,
                                 *[p(t) for t in x], p(wq), p(iold), p(delta), 1, None))
    _lib.check(L.smi_density_3d(2, p(want[3]), size, ints, (ctypes.c_double * 3)(*DX), 1.0, m, *[p(t) for t in x], p(wq),
                                None))
    torch.cuda.synchronize()
    for a, e in zip(got, want):
        assert float((a - e).abs().max()) <= 4e-13 * float(e.abs().max())
