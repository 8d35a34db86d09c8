"""Calls that take their scratch from the pool, from four host threads on four
streams at once and from one thread on three streams in turn: the results of
the same calls one at a time.

Currents add in another order each time: 1e-12 of the largest |J| (fewer than
2,000 contributions to a point); gathered fields and sorted particles are equal
bit for bit.  Sizes differ from thread to thread and from call to call, so that
the blocks of the pool change hands.
"""
import ctypes
import threading

import numpy as np
import pytest

from smilei_amd import _lib
from tests.test_gpu_binned_currents import DX, arrays, call, inputs

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


class Currents:
    def __init__(self, order, n, m, seed):
        self.order, self.n = order, n
        self.begin, self.dev, self.pos = inputs(order, n, m, "any", seed)
        self.J = arrays(order, n)
        self.start = [t.clone() for t in self.J]
        torch.cuda.synchronize()

    def go(self, stream):
        with torch.cuda.stream(stream):
            for t, s in zip(self.J, self.start):
                t.copy_(s)
            call(self.order, self.n, self.begin, self.dev, self.pos, 0, self.J, stream.cuda_stream)
            return [t.clone() for t in self.J]

    def same(self, a, b):
        return all(float((x - y).abs().max()) <= 1e-12 * float(y.abs().max()) for x, y in zip(a, b))


class Gather:
    def __init__(self, n, m, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        R = lambda s: torch.rand(s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
        self.np3, self.m = [v + 9 for v in n], m
        self.F = [R([self.np3[d] + ((c < 3) == (c % 3 == d)) for d in range(3)]) for c in range(6)]
        self.x = [R(m) * n[d] * DX[d] for d in range(3)]
        torch.cuda.synchronize()

    def go(self, stream):
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        I3, D3 = ctypes.c_int * 3, ctypes.c_double * 3
        with torch.cuda.stream(stream):
            E, B, d = (torch.zeros((3, self.m), dtype=torch.float64, device="cuda") for _ in range(3))
            i = torch.zeros((3, self.m), dtype=torch.int32, device="cuda")
            _lib.check(_lib.load().smi_interpolate_3d(4, *[p(t) for t in self.F], I3(*self.np3), I3(-4, -4, -4), D3(*DX),
                                                      self.m, *[p(t) for t in self.x], p(E), p(B), p(i), p(d),
                                                      ctypes.c_void_p(stream.cuda_stream)))
            return [E, B, i, d]

    def same(self, a, b):
        return all(torch.equal(x, y) for x, y in zip(a, b))


class Sort:
    def __init__(self, n, patch, m, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.n, self.patch, self.m = n, patch, m
        self.a = [torch.rand(m, generator=g, device="cuda", dtype=torch.float64) for _ in range(7)]
        for d in range(3):
            self.a[d] *= n[d] * DX[d]
        torch.cuda.synchronize()

    def go(self, stream):
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        I3, D3 = ctypes.c_int * 3, ctypes.c_double * 3
        with torch.cuda.stream(stream):
            a = [t.clone() for t in self.a]
            key = torch.zeros(self.m, dtype=torch.int32, device="cuda")
            _lib.check(_lib.load().smi_sort_exchange(3, I3(*self.n), I3(*self.patch), D3(*DX), self.m, *[p(t) for t in a],
                                                     None, p(key), None, None, ctypes.c_void_p(stream.cuda_stream)))
            return a + [key]

    same = Gather.same


def work():
    return [[Currents(2, (12, 13, 14), 20000, 1), Sort((16, 16, 16), (8, 8, 8), 70000, 2)],
            [Currents(4, (9, 8, 10), 3000, 3), Gather((10, 9, 8), 600000, 4)],
            [Currents(2, (40, 36, 44), 300000, 5), Currents(2, (8, 8, 8), 9000, 6)],
            [Sort((32, 16, 16), (8, 8, 8), 500000, 7), Currents(4, (12, 13, 14), 30000, 8)]]


def test_threads_and_streams():
    sets = work()
    alone = torch.cuda.Stream()
    want = [[w.go(alone) for w in s] for s in sets]
    torch.cuda.synchronize()
    failed = []

    def run(k):
        try:
            stream = torch.cuda.Stream()
            for _ in range(12):
                got = [w.go(stream) for w in sets[k]]
                stream.synchronize()
                failed.extend((k, j) for j, w in enumerate(sets[k]) if not w.same(got[j], want[k][j]))
            stream.synchronize()
        except Exception as e:  # noqa: BLE001 (reported by the test's own thread)
            failed.append((k, repr(e)))

    team = [threading.Thread(target=run, args=(k,)) for k in range(len(sets))]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not failed


def test_one_thread_several_streams():
    sets = [w for s in work() for w in s if not isinstance(w, Sort)]
    alone = torch.cuda.Stream()
    want = [w.go(alone) for w in sets]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    for _ in range(6):
        got = [w.go(streams[k % 3]) for k, w in enumerate(sets)]
        torch.cuda.synchronize()
        for w, a, b in zip(sets, got, want):
            assert w.same(a, b)
    assert np.isfinite(float(got[0][0].sum()))
