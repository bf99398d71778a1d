"""The radix sort under pxr_particle_bin_sorting and the binned leaf
routines, at the sizes where its blocks, waves and passes end, and the
binned direct current.

Bars: the sort moves values and is stable, so its output equals the oracle's
counting sort bit for bit.  The direct current sums the same FP64
contributions as the global-atomic form in another order: 1e-13 relative in
norm against it, 1e-12 against the oracle, as the other leaf depositions."""
import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, SHAPE, H, HG, T, TG, rel
from tests.test_gpu_leafbin import binned, dev, plasma, pxr  # noqa: F401

pytestmark = pytest.mark.gpu


# particles: one, a wave and a block of the sort with their neighbours, many
# blocks; bins: one (every key equal), one pass of digits, its edge at 2048,
# two passes, three (more than 2^22)
@pytest.mark.parametrize("n,cells", [
    (1, (5, 5, 5)), (63, (3, 2, 1)), (64, (1, 1, 1)), (65, (12, 9, 7)), (4095, (16, 16, 8)),
    (4096, (17, 11, 11)), (4097, (1, 1, 1)), (70001, (16, 16, 8)), (70001, (41, 50, 1)),
    (300007, (63, 64, 65)), (20011, (200, 170, 130)), (1023, (5, 5, 5)), (1024, (40, 9, 7)),
    (1025, (1, 1, 1)), (524287, (16, 16, 8)), (524288, (16, 16, 8)), (524288, (70, 50, 3))])
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


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("sort", [False, True])
def test_binned_direct_against_oracle_and_atomic_form(dev, pxr, orc, binned, order, sort):
    rng = np.random.default_rng(900 + order + 10 * sort)
    P, u, g, w, geo = plasma(rng, 120001, sort=sort, guard=0.5)
    xmin, ymin, zmin, dx, dy, dz = geo
    q, dt = -1.1, 0.45
    J0 = [np.asfortranarray(rng.standard_normal(SHAPE) * 0.1) for _ in range(3)]
    Jr = [j.copy(order="F") for j in J0]
    assert orc.depose_direct(*Jr, *P, *u, g, w, q, xmin, ymin, zmin, dt, dx, dy, dz, NX, NY, NZ,
                             NG, NG, NG, order) == 0
    out = []
    for bin_min in (1, 0):
        binned(bin_min)
        J = [TG(dev, j) for j in J0]
        pxr.depose_jxjyjz(*J, len(w), *[T(dev, a) for a in (*P, *u, g, w)], q, xmin, ymin, zmin,
                          dt, dx, dy, dz, NX, NY, NZ, NG, NG, NG, order, order, order, 3)
        out.append([HG(j) for j in J])
    for c in range(3):
        assert rel(out[0][c] - J0[c], Jr[c] - J0[c]) < 1e-12
        assert rel(out[0][c] - J0[c], out[1][c] - J0[c]) < 1e-13
