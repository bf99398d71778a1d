"""The scan of the radix sort's digit counts by one workgroup (up to 16384 of
them) and by many, at the sizes where one gives way to the other and where a
thread of the one workgroup takes another count.  Bit for bit against numpy's
stable sort of the same keys."""
import numpy as np
import pytest

from tests.test_gpu_leaf import H, T
from tests.test_gpu_leafbin import dev, pxr  # noqa: F401

pytestmark = pytest.mark.gpu


# counts = blocks of 1024 particles times 2^bits of the bins
@pytest.mark.parametrize("n,cells", [
    (8192, (16, 16, 8)), (8193, (16, 16, 8)), (1024, (16, 16, 4)), (1025, (16, 16, 4)),
    (16384, (16, 16, 4)), (16640, (16, 16, 4)), (65536, (16, 16, 1)), (66000, (16, 16, 1)),
    (500001, (2, 1, 1)), (7, (16, 16, 8))])
def test_counts_around_one_workgroup(dev, pxr, n, cells):  # noqa: F811
    rng = np.random.default_rng(n)
    P = [rng.uniform(0, c, n) for c in cells] + [rng.standard_normal(n) for _ in range(5)]
    key = (np.floor(P[2]) * cells[1] + np.floor(P[1])) * cells[0] + np.floor(P[0])
    o = np.argsort(key, kind="stable")
    D = [T(dev, p) for p in P]
    pxr.pxr_particle_bin_sorting(n, *D, 1, 0.0, 0.0, 0.0, *map(float, cells), 1.0, 1.0, 1.0)
    for d, p in zip(D, P):
        np.testing.assert_array_equal(H(d), p[o])
