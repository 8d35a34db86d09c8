"""smi_currents_3d's binning by one workgroup, by many with counts in LDS, and
with global counts, against the same call in index order.

Sizes on both sides of each line between the routes (8,192 and 12,288 particles
at order 2, 64 and 8,192 at order 4, 8,192 bins), one particle past a workgroup's
share, shuffled and in one bin.  Reordered sums and factorised weights of fewer
than 2,000 contributions to a point: 1e-12 of the largest |J|.
"""
import pytest

from tests.test_gpu_binned_currents import arrays, call, inputs

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("order,n,m,kind", [
    (2, (7, 9, 11), 8191, "any"), (2, (7, 9, 11), 8192, "any"), (2, (17, 9, 10), 12288, "cell order"),
    (2, (17, 9, 10), 12289, "strays"), (2, (24, 20, 24), 262145, "any"), (2, (24, 20, 24), 270001, "cell order"),
    (2, (40, 36, 44), 530000, "any"), (2, (75, 75, 75), 20001, "any"), (2, (76, 80, 78), 20001, "any"),
    (4, (4, 4, 4), 63, "any"), (4, (4, 4, 4), 64, "any"), (4, (8, 6, 7), 1025, "strays"), (4, (6, 8, 7), 700, "one bin"),
    (4, (16, 17, 18), 8192, "any"), (4, (16, 17, 18), 8193, "cell order")])
def test_routes(order, n, m, kind):
    begin, dev, pos = inputs(order, n, m, kind, 9)
    want, got = arrays(order, n), arrays(order, n)
    call(order, n, begin, dev, pos, 1, want)
    call(order, n, begin, dev, pos, 0, got)
    torch.cuda.synchronize()
    for a, b in zip(want, got):
        assert float((a - b).abs().max()) <= 1e-12 * float(a.abs().max())
