"""geteb3d_energy_conserving on sets in no order over enough blocks of a grid
that the library gathers them block by block from LDS (asserted): every shape,
one part and several, particles on the arrays' edges, outside them and not a
number.

Bar: an output is a sum of at most 4^3 field values with weights that add up
to one, so the forms differ by at most 70 roundings of the largest field value.
Particles outside the arrays are skipped and counted by both alike.
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_leaf import H, T, TG

pytestmark = pytest.mark.gpu

NG = 2
GRID = (80, 83, 78)  # 11 x 11 x 11 blocks
COUNTS = {1: (3145728, 8400001), 2: (786432,), 3: (786432, 8400001)}


@pytest.mark.parametrize("nodal", [0, 1])
@pytest.mark.parametrize("lower", [1, 0])
@pytest.mark.parametrize("order,n", [(o, n) for o in COUNTS for n in COUNTS[o]])
def test_staged_against_plain(order, n, lower, nodal):
    from picsar_amd import _lib
    _lib.call("pxrhip_init", 0)
    rng = np.random.default_rng(10 * order + 2 * lower + nodal)
    x = [rng.uniform(-1.0, g + 1.0, n) for g in GRID]
    for k, a in enumerate(x):
        a[rng.integers(0, n, 5)] = 1e4
        a[rng.integers(0, n, 5)] = -float(NG)
        a[rng.integers(0, n, 50)] = 8.0 * k + 6.0  # blocks' edges
        a[n // (k + 2)] = np.nan
    P = [T(_lib, a) for a in (0.3 + x[0] * 0.9, -1.0 + x[1], 2.0 + x[2] * 1.2)]
    F = [rng.standard_normal(tuple(g + 1 + 2 * NG for g in GRID)) for _ in range(6)]
    FD = [TG(_lib, f) for f in F]
    out = [rng.standard_normal(n) for _ in range(6)]
    old, form = C.c_int64(), C.c_int64()
    _lib.call("pxrhip_get_tuning", b"leaf.bin_min", C.byref(old))
    res = []
    try:
        for bin_min in (0, 1):
            _lib.call("pxrhip_set_tuning", b"leaf.bin_min", bin_min)
            e = [T(_lib, a) for a in out]
            with pytest.raises(_lib.PxrHipError, match="skipped") as err:
                _lib.call("pxrhip_geteb3d_energy_conserving", n, *[a.ptr for a in P],
                          *[a.ptr for a in e], 0.3, -1.0, 2.0, 0.9, 1.0, 1.2, *GRID, NG, NG, NG,
                          order, order, order, *[f.ptr for f in FD], 0, lower, 8, 0, nodal)
            _lib.call("pxrhip_get_tuning", b"last.leaf_gather", C.byref(form))
            assert form.value == bin_min
            res.append(([H(a) for a in e], str(err.value)))
    finally:
        _lib.call("pxrhip_set_tuning", b"leaf.bin_min", old.value)
    (a, ma), (b, mb) = res
    assert ma == mb
    eps = np.finfo(float).eps
    for f, p, q in zip(F, a, b):
        same = (p == q) | (np.isnan(p) & np.isnan(q))
        assert np.all(same | (np.abs(p - q) <= 70 * eps * np.abs(f).max() + eps * np.abs(p)))
