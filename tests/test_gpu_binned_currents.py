"""smi_currents_3d with free summation order against the same call in index
order, over the sizes where its routes change.

Both add the same contributions; the reordered sums, the factorised weights
and the left-out last face (a sum of DS over the whole window) move a point by
at most about (contributions) * 2^-53 * (largest contribution): fewer than
2,000 particles reach a point here, so 1e-12 of the largest |J| bounds it (the
bound of the operator tests).  Cases: below, at and above the size from which
particles are binned, in cell order and shuffled, ragged patches, all
particles in one bin (a full queue of node changers), particles whose stencil
leaves the arrays and particles that move two cells (both skipped), and a
captured call (no scratch) next to an ordinary one.
"""
import ctypes

import numpy as np
import pytest

from smilei_amd import _lib
from tests.plasma import cfl_dt

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DX = (0.2, 0.25, 0.3)


def inputs(order, n, m, kind, seed):
    """Old nodes, offsets, new positions and weights of m particles of a
    patch of n cells whose first cell is global cell (8, 4, 0)."""
    rng = np.random.default_rng(seed)
    first = np.array([8, 4, 0])
    cells = np.stack([rng.integers(0, n[d], m) for d in range(3)])
    if kind == "one bin":
        cells = np.tile(np.array([[3], [1], [2]]), (1, m))
    if kind == "cell order":
        cells = cells[:, np.lexsort(cells[::-1])]
    pn = first[:, None] + cells + rng.random((3, m))
    node = np.floor(pn + 0.5)
    move = rng.uniform(-0.9, 0.9, (3, m)) * (rng.random(m) < (0.9 if kind == "one bin" else 0.3))
    if kind == "strays":
        move[0, ::7] = 2.5  # more than one cell
    iold = (node - first[:, None] + order).astype(np.int32)
    if kind == "strays":
        iold[1, ::11] = 0  # no room for the stencil
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (iold, pn - node, rng.random(m) + 0.5)]
    pos = [torch.from_numpy((pn[d] + move[d]) * DX[d]).cuda() for d in range(3)]
    return first - order, dev, pos


def call(order, n, begin, dev, pos, deterministic, J, stream=0):
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    ints = lambda v: (ctypes.c_int * 3)(*[int(a) for a in v])  # noqa: E731
    _lib.check(_lib.load().smi_currents_3d(order, *[p(t) for t in J], ints([v + 2 * order + 1 for v in n]), ints(begin),
                                           (ctypes.c_double * 3)(*DX), cfl_dt(DX), -1.5, len(dev[2]),
                                           *[p(t) for t in pos], p(dev[2]), p(dev[0]), p(dev[1]), deterministic,
                                           ctypes.c_void_p(stream)))


def arrays(order, n, seed=1):
    """Currents that already hold something: the call adds to them."""
    g = torch.Generator().manual_seed(seed)
    return [torch.rand([n[d] + 2 * order + 1 + (d == c) for d in range(3)], generator=g, dtype=torch.float64).cuda()
            for c in range(3)]


@pytest.mark.parametrize("order,n,m,kind", [
    (2, (6, 9, 11), 12287, "any"), (2, (6, 9, 11), 12288, "any"), (2, (21, 8, 13), 20000, "cell order"),
    (2, (8, 8, 8), 14000, "one bin"), (2, (9, 10, 7), 15000, "strays"), (4, (5, 9, 11), 511, "any"),
    (4, (5, 9, 11), 512, "any"), (4, (13, 8, 9), 6000, "cell order"), (4, (8, 8, 8), 1500, "one bin"),
    (4, (9, 7, 10), 3000, "strays")])
def test_same_currents_as_in_index_order(order, n, m, kind):
    begin, dev, pos = inputs(order, n, m, kind, 5)
    want, got = arrays(order, n), arrays(order, n)
    call(order, n, begin, dev, pos, 1, want)
    call(order, n, begin, dev, pos, 0, got)
    torch.cuda.synchronize()
    for a, b in zip(want, got):
        assert float((a - b).abs().max()) <= 1e-12 * float(a.abs().max())


def test_captured_call():
    n, order, m = (9, 8, 10), 2, 16000
    begin, dev, pos = inputs(order, n, m, "any", 6)
    want, got = arrays(order, n), arrays(order, n)
    keep = [t.clone() for t in got]
    call(order, n, begin, dev, pos, 0, want)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call(order, n, begin, dev, pos, 0, got, s.cuda_stream)
    for _ in range(3):
        for t, k in zip(got, keep):
            t.copy_(k)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(want, got):
            assert float((a - b).abs().max()) <= 1e-12 * float(a.abs().max())
