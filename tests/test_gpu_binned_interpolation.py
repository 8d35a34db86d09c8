"""smi_interpolate_3d over binned particles against the same particles in calls
too small to be binned: the same bits.

5.2e5 particles and more at order 4 are binned where there are 160 to a bin; the
products and sums are those of the direct gather.  Sizes at the line, one past
it, patches that are no multiple of four, particles in cell order, shuffled, in
one corner, and a fifth of them outside the patch (NaN, and no node written).
"""
import ctypes

import numpy as np
import pytest

from smilei_amd import _lib

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DX = (0.2, 0.25, 0.3)
M = 1 << 19


def call(np3, begin, F, pos, lo, hi):
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    I3, D3 = ctypes.c_int * 3, ctypes.c_double * 3
    m = hi - lo
    x = [t[lo:hi].contiguous() for t in pos]
    E, B = (torch.full((3, m), 7.0, dtype=torch.float64, device="cuda") for _ in range(2))
    iold = torch.full((3, m), -5, dtype=torch.int32, device="cuda")
    delta = torch.full((3, m), 9.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    _lib.check(_lib.load().smi_interpolate_3d(4, *[p(t) for t in F], I3(*np3), I3(*begin), D3(*DX), m,
                                              *[p(t) for t in x], p(E), p(B), p(iold), p(delta), None))
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in (E, B, iold, delta)]


@pytest.mark.parametrize("n,m,kind", [((12, 13, 18), M, "any"), ((12, 13, 18), M + 1, "cell order"),
                                      ((37, 38, 39), M + 77777, "any"), ((9, 6, 7), M + 3, "corner"),
                                      ((21, 30, 17), M + 1000, "outside"), ((88, 88, 88), 2200000, "any")])
def test_same_bits(n, m, kind):
    rng = np.random.default_rng(m)
    order, first = 4, (8, 4, 0)
    np3 = [v + 2 * order + 1 for v in n]
    begin = [f - order for f in first]
    F = [torch.from_numpy(rng.standard_normal([np3[d] + ((c < 3) == (c % 3 == d)) for d in range(3)])).cuda()
         for c in range(6)]
    cells = [rng.integers(0, 3 if kind == "corner" else n[d], m) for d in range(3)]
    if kind == "cell order":
        o = np.lexsort(cells[::-1])
        cells = [c[o] for c in cells]
    pos = [(first[d] + cells[d] + rng.random(m)) * DX[d] for d in range(3)]
    if kind == "outside":
        far = rng.random(m) < 0.2
        pos[1] = np.where(far, pos[1] + (n[1] + 5) * DX[1] * rng.choice([-1, 1], m), pos[1])
    pos = [torch.from_numpy(v).cuda() for v in pos]
    got = call(np3, begin, F, pos, 0, m)
    step = 400000
    parts = [call(np3, begin, F, pos, lo, min(lo + step, m)) for lo in range(0, m, step)]
    for k in range(4):
        want = np.concatenate([q[k] for q in parts], axis=1)
        assert np.array_equal(got[k], want, equal_nan=k != 2)
    assert np.isnan(got[0]).any() == (kind == "outside")
