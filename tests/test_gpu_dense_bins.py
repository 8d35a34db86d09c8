"""Currents and densities of the binned device projector with many particles
per cell: the cell-sorted walk against the strided one (the same contributions
in another order), and its time.

Fewer than 20,000 particles reach a point and each contribution is the same in
both walks; they drift one way, so the sums differ by at most 2 * 20,000 * 2^-53
of the largest |value|.  Both sides of 128 bins, where the length of a thread's
run changes, ragged bins, empty ones, and one particle.  Four times as many
particles in 4,096 bins take less than seven times as long (4.8 times; with
one run per thread 9.3, its lines leaving the caches between two particles).
"""
import ctypes

import pytest

from smilei_amd import _lib

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DX, DT, F64 = (0.2, 0.25, 0.3), 0.1, torch.float64


def inputs(nb, counts, seed=3):
    g = torch.Generator(device="cuda").manual_seed(seed)
    bins = nb[0] * nb[1] * nb[2]
    n = [4 * v for v in nb]
    count = torch.tensor([counts[b % len(counts)] for b in range(bins)], device="cuda")
    ends = torch.cumsum(count, 0).to(torch.int32)
    m = int(ends[-1])
    b = torch.repeat_interleave(torch.arange(bins, device="cuda"), count)
    at = torch.arange(m, device="cuda") - (torch.cumsum(count, 0) - count)[b]
    cell = (64 * at) // count[b]  # in cell order inside a bin
    low = [(b // (nb[1] * nb[2])) * 4 + cell // 16, (b // nb[2]) % nb[1] * 4 + (cell // 4) % 4, b % nb[2] * 4 + cell % 4]
    pn = [low[d] + torch.rand(m, generator=g, device="cuda", dtype=F64) for d in range(3)]
    node = [torch.round(v) for v in pn]
    return dict(nb=list(nb), n=n, m=m, ends=ends, iold=torch.stack([v + 2 for v in node]).to(torch.int32),
                delta=torch.stack([pn[d] - node[d] for d in range(3)]),
                new=[(pn[d] + 0.2 * torch.rand(m, generator=g, device="cuda", dtype=F64)) * DX[d] for d in range(3)],
                w=0.5 + torch.rand(m, generator=g, device="cuda", dtype=F64), invgf=torch.ones(m, device="cuda", dtype=F64),
                charge=torch.ones(m, device="cuda", dtype=torch.int16))


def deposit(s, cell_sorting):
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    L, n = _lib.load(), s["n"]
    out = [torch.zeros([n[d] + 5 + (d == c) for d in range(3)], device="cuda", dtype=F64) for c in range(4)]
    torch.cuda.synchronize()
    tail = ([p(t) for t in s["new"]] + [p(s["charge"]), p(s["w"]), p(s["ends"])] + s["nb"]
            + [p(s["invgf"]), p(s["iold"]), p(s["delta"]), s["m"], 1.0] + [1.0 / v for v in DX] + [v / DT for v in DX]
            + [-2, -2, -2, n[1] + 5, n[2] + 5, 1, cell_sorting])
    _lib.check(L.smi_current_deposition_3d(*[p(t) for t in out[:3]], *[t.numel() for t in out[:3]], *tail))
    _lib.check(L.smi_density_deposition_3d(p(out[3]), out[3].numel(), *tail))
    return out


@pytest.mark.parametrize("nb,counts", [((4, 4, 8), [5000, 0, 1, 4097]), ((4, 4, 9), [1024, 1025, 1023, 1, 0, 5000]),
                                       ((6, 6, 6), [4096, 1500, 300])])
def test_both_walks_agree(nb, counts):
    s = inputs(nb, counts)
    for a, b in zip(deposit(s, True), deposit(s, False)):
        assert float((a - b).abs().max()) <= 2 * 20000 * 2.0 ** -53 * float(b.abs().max())


def test_time_grows_with_the_particles():
    import time
    times = []
    for count in (1024, 4096):
        s = inputs((16, 16, 16), [count])
        deposit(s, True)
        runs = []
        for _ in range(5):
            t = time.perf_counter()
            deposit(s, True)
            runs.append(time.perf_counter() - t)
        times.append(sorted(runs)[2])
    assert times[1] <= 7 * times[0]
