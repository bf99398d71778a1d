"""geteb3d_energy_conserving on large particle sets: one in no order is
gathered block by block from LDS, one in cell order from the grid arrays.

Bar: an output is a sum of at most 4^3 field values with weights that add up
to one, so the forms (and any contraction of their products) differ by at
most 70 roundings of the largest field value.  Particles outside the arrays
are skipped and counted by both alike.
"""
import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, SHAPE, H, T, TG, particles

pytestmark = pytest.mark.gpu

COUNTS = {1: (3145727, 3145728), 2: (786431, 786432, 1700001),
          3: (786431, 786432, 900001, 8400001)}


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


def gather(dev, pxr, P, F, out, order, lower, bin_min):
    from picsar_amd import _lib
    import ctypes
    old = ctypes.c_int64()
    _lib.call("pxrhip_get_tuning", b"leaf.bin_min", ctypes.byref(old))
    _lib.call("pxrhip_set_tuning", b"leaf.bin_min", bin_min)
    o = [T(dev, a) for a in out]
    msg = ""
    try:
        pxr.geteb3d_energy_conserving(len(P[0]), *P, *o, 0.3, -1.0, 2.0, 0.9, 1.0, 1.2, NX, NY, NZ,
                                      NG, NG, NG, order, order, order, *F, False, lower)
    except _lib.PxrHipError as e:
        msg = str(e)
    finally:
        _lib.call("pxrhip_set_tuning", b"leaf.bin_min", old.value)
    return [H(a) for a in o], msg


@pytest.mark.parametrize("nodal", [False, True])
@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("order,n", [(o, n) for o in COUNTS for n in COUNTS[o]])
def test_sets_in_no_order(dev, order, n, lower, nodal):
    from picsar_amd.picsarpy import picsar
    rng = np.random.default_rng(order * 100 + lower)
    x, y, z = particles(rng, n, lo=-1.0, margin=0.0)
    for k, a in enumerate((x, y, z)):  # outside the arrays, on their edge, and not a number
        a[rng.integers(0, n, 5)] = 1e4
        a[rng.integers(0, n, 5)] = -float(NG)
    x[n // 3] = y[n // 2] = z[-1] = np.nan
    P = [T(dev, a) for a in (0.3 + x * 0.9, -1.0 + y, 2.0 + z * 1.2)]
    F = [rng.standard_normal(SHAPE) for _ in range(6)]
    FD = [TG(dev, f) for f in F]
    out = [rng.standard_normal(n) for _ in range(6)]
    out[2][:100] = -0.0
    was = picsar.l_nodalgrid
    picsar.l_nodalgrid = nodal
    try:
        a, ma = gather(dev, picsar, P, FD, out, order, lower, 0)
        b, mb = gather(dev, picsar, P, FD, out, order, lower, 1)
    finally:
        picsar.l_nodalgrid = was
    assert ma == mb and "skipped" in ma
    for f, p, q in zip(F, a, b):
        tol = 70 * np.finfo(float).eps * np.abs(f).max() + np.finfo(float).eps * np.abs(p)
        same = (p == q) | (np.isnan(p) & np.isnan(q))
        assert np.all(same | (np.abs(p - q) <= tol))


@pytest.mark.parametrize("swap", [0, 20])
def test_sets_in_cell_order(dev, swap):
    """cell order, also with a few particles exchanged, keeps the plain form"""
    from picsar_amd.picsarpy import picsar
    rng = np.random.default_rng(5)
    n = 800000
    x, y, z = particles(rng, n, lo=0.0, margin=1.0)
    o = np.lexsort((np.floor(x), np.floor(y), np.floor(z)))
    i, j = rng.integers(0, n, swap), rng.integers(0, n, swap)
    o[i], o[j] = o[j].copy(), o[i].copy()
    P = [T(dev, a[o]) for a in (0.3 + x * 0.9, -1.0 + y, 2.0 + z * 1.2)]
    FD = [TG(dev, rng.standard_normal(SHAPE)) for _ in range(6)]
    out = [np.zeros(n) for _ in range(6)]
    a, _ = gather(dev, picsar, P, FD, out, 3, True, 0)
    b, _ = gather(dev, picsar, P, FD, out, 3, True, 1)
    for p, q in zip(a, b):
        np.testing.assert_array_equal(p, q)


def test_calls_of_several_threads(dev):
    """The library's stream and scratch are shared: calls of several threads
    give what they give one after the other."""
    import threading
    from picsar_amd.picsarpy import picsar
    rng = np.random.default_rng(11)
    n = 800000
    FD = [TG(dev, rng.standard_normal(SHAPE)) for _ in range(6)]
    sets = []
    for k in range(3):
        x, y, z = particles(rng, n, margin=1.0)
        if k == 1:
            o = np.lexsort((np.floor(x), np.floor(y), np.floor(z)))
            x, y, z = x[o], y[o], z[o]
        sets.append([T(dev, a) for a in (x, y, z)])
    outs = [[[T(dev, np.zeros(n)) for _ in range(6)] for _ in range(4)] for _ in sets]

    def run(k, r):
        picsar.geteb3d_energy_conserving(n, *sets[k], *outs[k][r], 0.0, 0.0, 0.0, 1.0, 1.0, 1.0,
                                         NX, NY, NZ, NG, NG, NG, 3, 3, 3, *FD, False, True)

    was, picsar.l_nodalgrid = picsar.l_nodalgrid, False
    try:
        for k in range(3):
            run(k, 0)
        th = [threading.Thread(target=lambda k=k: [run(k, r) for r in (1, 2, 3)]) for k in range(3)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    finally:
        picsar.l_nodalgrid = was
    for k in range(3):
        for r in (1, 2, 3):
            for a, b in zip(outs[k][0], outs[k][r]):
                np.testing.assert_array_equal(H(a), H(b))
