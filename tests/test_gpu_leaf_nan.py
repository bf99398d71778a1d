"""Particles whose position is not a number in the binned leaf depositions.
The library's index of such a coordinate is node 0; their block is the first,
which does not reach node 0 where the guards are wide, and they are then added
to the grid arrays directly.  Both forms leave the same nodes not a number and
agree on the others up to n roundings of the largest node (another order of
the sums).
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_leaf import HG, T, TG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("guard", [3, 12])
@pytest.mark.parametrize("order", [1, 2, 3])
def test_nan_positions(order, guard):
    from picsar_amd import _lib
    _lib.call("pxrhip_init", 0)
    n, grid = 4001, (20, 18, 14)
    rng = np.random.default_rng(order)
    x = [rng.uniform(3.0, g - 3.0, n) for g in grid]
    x[0][7] = x[1][100] = x[2][2000] = x[0][300] = x[1][300] = np.nan
    u = [rng.uniform(-0.5, 0.5, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    P = [T(_lib, a) for a in (*x, *u, g, rng.uniform(0.5, 2.0, n))]
    shape = tuple(c + 1 + 2 * guard for c in grid)
    old, form = C.c_int64(), C.c_int64()
    _lib.call("pxrhip_get_tuning", b"leaf.bin_min", C.byref(old))
    out = []
    try:
        for bin_min in (0, 1):
            _lib.call("pxrhip_set_tuning", b"leaf.bin_min", bin_min)
            res = []
            for algo in (0, 3):
                J = [TG(_lib, np.zeros(shape)) for _ in range(3)]
                _lib.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in P], -1.1,
                          0.0, 0.0, 0.0, 0.4, 1.0, 1.0, 1.0, *grid, guard, guard, guard, order,
                          order, order, algo, 0)
                _lib.call("pxrhip_get_tuning", b"last.leaf_current", C.byref(form))
                assert form.value == bin_min
                res += [HG(j) for j in J]
            r = TG(_lib, np.zeros(shape))
            _lib.call("pxrhip_depose_rho_n", r.ptr, n, *[P[k].ptr for k in (0, 1, 2, 7)], -1.1, 0.0,
                      0.0, 0.0, 1.0, 1.0, 1.0, *grid, guard, guard, guard, order, order, order, 1, 0)
            _lib.call("pxrhip_get_tuning", b"last.leaf_rho", C.byref(form))
            assert form.value == bin_min
            out.append(res + [HG(r)])
    finally:
        _lib.call("pxrhip_set_tuning", b"leaf.bin_min", old.value)
    for a, b in zip(*out):
        assert np.isnan(a).any() and not np.isnan(a).all()
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
        ok = ~np.isnan(a)
        assert np.abs(a - b)[ok].max() <= n * np.finfo(float).eps * np.abs(a[ok]).max()
