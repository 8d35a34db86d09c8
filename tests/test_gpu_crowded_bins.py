"""Binned operators where most particles lie in a few bins: crowded bins are
worked on in shares of 1,024 particles (more from 2.1e6 particles on).

Currents against the same call in index order: the particles drift one way,
so that the contributions to a point have one sign and the reordered sum of m
of them, each rounded a few tens of times, moves it by at most (2 m + 100) *
2^-53 of the largest |J|.  Fields gathered by position: the same bits as in calls
too small to be binned.  Crowds one below, at and above one and two shares, in
each binning route (one workgroup, counts in LDS, global counts).  And the
times: a crowd takes no more than eight times as long as the same particles
spread over the patch (0.4 to 1.5 times with shares, 19 to 190 with one
workgroup per bin).
"""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_binned_currents import DX, arrays, call
from tests.test_gpu_binned_interpolation import call as gather

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def drifting(order, n, m, crowd, seed=4):
    """m particles of a patch of n cells, `crowd` of them in each of two cells."""
    rng = np.random.default_rng(seed)
    first = np.array([8, 4, 0])
    cells = np.stack([rng.integers(0, n[d], m) for d in range(3)])
    cells[:, :crowd] = [[2], [5], [1]]
    cells[:, crowd:2 * crowd] = [[5], [2], [4]]
    cells = cells[:, rng.permutation(m)]
    pn = first[:, None] + cells + rng.random((3, m))
    node = np.floor(pn + 0.5)
    iold = (node - first[:, None] + order).astype(np.int32)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (iold, pn - node, rng.random(m) + 0.5)]
    pos = [torch.from_numpy((pn[d] + 0.1 + 0.2 * rng.random(m)) * DX[d]).cuda() for d in range(3)]
    return first - order, dev, pos


@pytest.mark.parametrize("order,n,m,crowd", [
    (2, (8, 9, 7), 9000, 1023), (2, (8, 9, 7), 9000, 1024), (2, (8, 9, 7), 9000, 1025), (2, (12, 9, 8), 16000, 2049),
    (2, (9, 10, 8), 30000, 14000), (2, (76, 80, 78), 24000, 6000), (4, (8, 9, 7), 2500, 1024), (4, (8, 9, 7), 2500, 1025),
    (4, (12, 9, 8), 12000, 5000)])
def test_crowded_currents(order, n, m, crowd):
    begin, dev, pos = drifting(order, n, m, crowd)
    want, got = arrays(order, n), arrays(order, n)
    call(order, n, begin, dev, pos, 1, want)
    call(order, n, begin, dev, pos, 0, got)
    torch.cuda.synchronize()
    for a, b in zip(want, got):
        assert float((a - b).abs().max()) <= (2 * m + 100) * 2.0 ** -53 * float(a.abs().max())


def fields(np3, seed=2):
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.standard_normal([np3[d] + ((c < 3) == (c % 3 == d)) for d in range(3)])).cuda()
            for c in range(6)]


def test_larger_shares_gather_the_same_bits():
    n, m, first = (9, 6, 7), 3000001, (8, 4, 0)
    rng = np.random.default_rng(3)
    np3 = [v + 9 for v in n]
    F = fields(np3)
    cell = [rng.integers(0, 2, m) for _ in range(3)]
    pos = [torch.from_numpy((first[d] + 4 + cell[d] + rng.random(m)) * DX[d]).cuda() for d in range(3)]
    begin = [f - 4 for f in first]
    got = gather(np3, begin, F, pos, 0, m)
    step = 400000
    parts = [gather(np3, begin, F, pos, lo, min(lo + step, m)) for lo in range(0, m, step)]
    for k in range(4):
        assert np.array_equal(got[k], np.concatenate([q[k] for q in parts], axis=1))


def duration(go):
    """Median of five, in ms."""
    times = []
    for _ in range(6):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        go()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    return sorted(times[1:])[2]


@pytest.mark.parametrize("order", [2, 4])
def test_a_crowd_of_currents_fills_the_chip(order):
    n, m = (32, 32, 32), 300000
    times = []
    for crowd in (0, m // 2):
        begin, dev, pos = drifting(order, n, m, crowd)
        J = arrays(order, n)
        stream = torch.cuda.current_stream().cuda_stream
        times.append(duration(lambda: call(order, n, begin, dev, pos, 0, J, stream)))
    assert times[1] <= 8 * times[0]


def test_a_crowd_of_gathers_fills_the_chip():
    from smilei_amd import _lib
    n, m, np3, first = (32, 32, 32), 600000, [41, 41, 41], (8, 4, 0)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    I3, D3 = ctypes.c_int * 3, ctypes.c_double * 3
    F, rng, times = fields(np3), np.random.default_rng(5), []
    E, B, delta = (torch.empty((3, m), dtype=torch.float64, device="cuda") for _ in range(3))
    iold = torch.empty((3, m), dtype=torch.int32, device="cuda")
    for width in (32, 2):
        x = [torch.from_numpy((first[d] + width * rng.random(m)) * DX[d]).cuda() for d in range(3)]
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        times.append(duration(lambda: _lib.check(_lib.load().smi_interpolate_3d(
            4, *[p(t) for t in F], I3(*np3), I3(*[f - 4 for f in first]), D3(*DX), m, *[p(t) for t in x], p(E), p(B),
            p(iold), p(delta), stream))))
    assert times[1] <= 8 * times[0]
