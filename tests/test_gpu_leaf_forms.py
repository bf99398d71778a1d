"""Which form a large leaf call takes, as the library reports it: sets in no
order and in cell order, sizes on both sides of each rule, sets ordered in
several parts.  Results are compared in the tests of the forms themselves.
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, SHAPE, T, TG, particles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


def last(dev, what):
    v = C.c_int64()
    dev.call("pxrhip_get_tuning", b"last.leaf_" + what, C.byref(v))
    return v.value


def cell_order(x):
    return np.lexsort(tuple(np.floor(a) for a in x))


def plasma(dev, n, grid, ordered):
    rng = np.random.default_rng(n)
    x = particles(rng, n, margin=1.0) if grid is None else [rng.uniform(1, g - 1, n) for g in grid]
    if ordered:
        o = cell_order(x)
        x = [a[o] for a in x]
    u = [rng.uniform(-1.0, 1.0, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    return [T(dev, a) for a in (*x, *u, g, rng.uniform(0.5, 2.0, n))]


def gather(dev, n, x, order, grid=(NX, NY, NZ), lower=1):
    shape = tuple(g + 1 + 2 * NG for g in grid)
    F = TG(dev, np.zeros(shape))
    e = T(dev, np.zeros(n))
    dev.call("pxrhip_geteb3d_energy_conserving", n, *[a.ptr for a in x], *[e.ptr] * 6, 0.0, 0.0,
             0.0, 1.0, 1.0, 1.0, *grid, NG, NG, NG, order, order, order, *[F.ptr] * 6, 0, lower, 8,
             0, 0)
    return last(dev, b"gather")


def current(dev, n, P, order, algo, grid=(NX, NY, NZ)):
    J = [TG(dev, np.zeros(tuple(g + 1 + 2 * NG for g in grid))) for _ in range(3)]
    dev.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in P], -1.1, 0.0, 0.0,
             0.0, 0.3, 1.0, 1.0, 1.0, *grid, NG, NG, NG, order, order, order, algo, 0)
    return last(dev, b"current"), last(dev, b"records")


BIG = (100, 100, 100)  # 2744 blocks


@pytest.mark.parametrize("order,n,form", [
    (1, 3145727, 0), (1, 3145728, 1), (2, 786431, 0), (2, 786432, 1), (3, 786431, 0),
    (3, 786432, 1), (3, 8400001, 1)])
@pytest.mark.parametrize("ordered", [False, True])
def test_gather(dev, order, n, form, ordered):
    x = plasma(dev, n, BIG, ordered)[:3]
    assert gather(dev, n, x, order, BIG) == (0 if ordered else form)


@pytest.mark.parametrize("exchanged,form", [(20, 0), (900000, 1)])
def test_gather_of_a_set_losing_its_order(dev, exchanged, form):
    """a few particles exchanged, and most of them"""
    n = 900000
    rng = np.random.default_rng(exchanged)
    x = [rng.uniform(1, g - 1, n) for g in BIG]
    o = cell_order(x)
    i = rng.permutation(n)[:exchanged]
    o[i] = o[np.roll(i, 1)]
    assert gather(dev, n, [T(dev, a[o]) for a in x], 3, BIG) == form


@pytest.mark.parametrize("algo", [0, 3])
@pytest.mark.parametrize("order,n,records", [
    (1, 524287, 0), (1, 524288, 1), (2, 524288, 1), (2, 8388609, 1), (3, 524288, 0)])
@pytest.mark.parametrize("ordered", [False, True])
def test_records(dev, order, n, records, algo, ordered):
    P = plasma(dev, n, None, ordered)
    assert current(dev, n, P, order, algo) == (1, 0 if ordered else records)


@pytest.mark.parametrize("n,form", [(65535, 0), (65536, 1)])
def test_depositions(dev, n, form):
    P = plasma(dev, n, None, False)
    for algo in (0, 3):
        assert current(dev, n, P, 1, algo) == (form, 0)
    r = TG(dev, np.zeros(SHAPE))
    dev.call("pxrhip_depose_rho_n", r.ptr, n, *[P[k].ptr for k in (0, 1, 2, 7)], -1.1, 0.0, 0.0,
             0.0, 1.0, 1.0, 1.0, NX, NY, NZ, NG, NG, NG, 1, 1, 1, 1, 0)
    assert last(dev, b"rho") == form


@pytest.mark.parametrize("order,grid,n,form", [
    # 26^3 = 17576, 35^3 = 42875 and 65 x 65 x 9 = 38025 blocks
    (1, (200, 200, 200), 192 * 17576 - 1, 0), (1, (200, 200, 200), 192 * 17576, 1),
    (2, (200, 200, 200), 48 * 17576 - 1, 0), (2, (200, 200, 200), 48 * 17576, 1),
    (3, (270, 270, 270), 24 * 42875 - 1, 0), (3, (270, 270, 270), 24 * 42875, 1),
    (3, (512, 512, 64), 24 * 38025 - 1, 0), (3, (512, 512, 64), 24 * 38025, 1)])
def test_gather_on_a_sparse_grid(dev, order, grid, n, form):
    """the blocks' fields are staged only where enough particles read them"""
    rng = np.random.default_rng(n)
    assert gather(dev, n, [T(dev, rng.uniform(1, g - 1, n)) for g in grid], order, grid) == form


def block_counts(x, grid):
    b = [(np.floor(a).astype(int) + NG) // 8 for a in x]
    nb = [-(-(g + 1 + 2 * NG) // 8) for g in grid]
    return np.bincount(b[0] + nb[0] * (b[1] + nb[1] * b[2]))


@pytest.mark.parametrize("chunk", [1, 100, 512, 4096, 4097, 30000, 1 << 20])
def test_work_items(dev, chunk):
    """leaf.bin_chunk bounds the work items and, above its default, sets them"""
    n, grid = 70001, (NX, NY, NZ)
    rng = np.random.default_rng(chunk)
    x = particles(rng, n, margin=1.0)
    x[0][: n // 2] = rng.uniform(6, 10, n // 2)
    P = [T(dev, a) for a in (*x, *np.zeros((3, n)), np.ones(n), np.ones(n))]
    c = block_counts(x, grid)
    old = C.c_int64()
    dev.call("pxrhip_get_tuning", b"leaf.bin_chunk", C.byref(old))
    assert old.value == 4096
    try:
        dev.call("pxrhip_set_tuning", b"leaf.bin_chunk", chunk)
        for order, algo, own in ((1, 0, 512), (2, 3, 1024), (3, 0, 2048)):
            assert current(dev, n, P, order, algo) == (1, 0)
            size = chunk if chunk > 4096 else min(chunk, own)
            assert last(dev, b"items") == (-(-c // size)).sum()
    finally:
        dev.call("pxrhip_set_tuning", b"leaf.bin_chunk", old.value)


@pytest.mark.parametrize("n,direct", [(17575, 0), (17576, 0), (8 * 17576 - 1, 0), (8 * 17576, 1)])
def test_currents_on_a_sparse_grid(dev, n, direct):
    """26^3 = 17576 blocks: one particle each for Esirkepov, eight for direct"""
    grid = (200, 200, 200)
    P = plasma(dev, n, grid, False)
    old = C.c_int64()
    dev.call("pxrhip_get_tuning", b"leaf.bin_min", C.byref(old))
    try:
        dev.call("pxrhip_set_tuning", b"leaf.bin_min", 1)
        assert current(dev, n, P, 1, 0, grid)[0] == (n >= 17576)
        assert current(dev, n, P, 1, 3, grid)[0] == direct
    finally:
        dev.call("pxrhip_set_tuning", b"leaf.bin_min", old.value)


@pytest.mark.parametrize("order,n,sigma,form", [
    (1, 4000000, 3.0, 0), (1, 4000000, 12.0, 0), (1, 4000000, 30.0, 1), (2, 1000000, 3.0, 0),
    (2, 1000000, 24.0, 1), (2, 4000000, 1.5, 0), (2, 4000000, 12.0, 1), (3, 1000000, 1.5, 0),
    (3, 1000000, 12.0, 1), (3, 4000000, 3.0, 1)])
def test_gather_of_a_bunch(dev, order, n, sigma, form):
    """particles in few blocks are gathered plainly, whatever their order"""
    grid = (128, 128, 128)
    rng = np.random.default_rng(int(10 * sigma))
    x = [np.clip(rng.normal(0.6 * g, sigma, n), 1.0, g - 1.0) for g in grid]
    assert gather(dev, n, [T(dev, a) for a in x], order, grid) == form
