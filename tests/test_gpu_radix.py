"""The radix sort under pxr_particle_bin_sorting, at the sizes where its
blocks, waves and passes end.  It moves values and is stable, so its output
equals the oracle's counting sort bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_leaf import H, T, dev, pxr  # noqa: F401

pytestmark = pytest.mark.gpu


# particles: one, a wave and a block of the sort with their neighbours, many
# blocks; bins: one (every key equal), one pass of digits, its edge at 2048,
# two passes, three (more than 2^22)
@pytest.mark.parametrize("n,cells", [
    (1, (5, 5, 5)), (63, (3, 2, 1)), (64, (1, 1, 1)), (65, (12, 9, 7)), (4095, (16, 16, 8)),
    (4096, (17, 11, 11)), (4097, (1, 1, 1)), (70001, (16, 16, 8)), (70001, (41, 50, 1)),
    (300007, (63, 64, 65)), (20011, (200, 170, 130))])
def test_sort_sizes_bitexact(dev, pxr, orc, n, cells):
    rng = np.random.default_rng(n + cells[0])
    P = [rng.uniform(0, c, n) for c in cells] + [rng.standard_normal(n) for _ in range(4)]
    P.append(np.arange(n, dtype=np.float64))
    box = (0.0, 0.0, 0.0, *map(float, cells), 1.0, 1.0, 1.0)
    Q = [p.copy() for p in P]
    assert orc.particle_bin_sorting(*Q, *box) == 0
    D = [T(dev, p) for p in P]
    pxr.pxr_particle_bin_sorting(n, *D, 1, *box)
    for a, b in zip(D, Q):
        np.testing.assert_array_equal(H(a), b)

