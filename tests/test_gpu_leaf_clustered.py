"""Large leaf calls whose particles sit in few blocks of a large grid, all in
one block, or evenly: the work items of blocks without particles, of blocks
with a few, and of one that a whole wave cuts up; block counts on both sides of
what one pass of the sort takes (2048), set sizes on both sides of those whose
keys are counted as they are made (2^19).

Against the unbinned form on the same particles: a node's sum has at most n
terms, added in another order, so the bar is n roundings of the largest node.
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_leaf import HG, T, TG, H

pytestmark = pytest.mark.gpu

NG = 3
# 8^3-node blocks of the padded grid: 125, 2040, 2197, 8000
GRIDS = ((32, 32, 32), (127, 113, 56), (97, 97, 97), (150, 150, 150))


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


def positions(rng, n, grid, kind):
    if kind == "even":
        return [rng.uniform(1.0, g - 1.0, n) for g in grid]
    if kind == "bunch":
        return [np.clip(rng.normal(0.6 * g, 2.0, n), 1.0, g - 1.0) for g in grid]
    # inside one block: nodes 8 m - 3 .. 8 m + 4
    return [8 * (g // 16) - 3 + rng.uniform(2.0, 6.0, n) for g in grid]


def both(dev, fn):
    old = C.c_int64()
    dev.call("pxrhip_get_tuning", b"leaf.bin_min", C.byref(old))
    out = []
    try:
        for bin_min in (0, 1):
            dev.call("pxrhip_set_tuning", b"leaf.bin_min", bin_min)
            out.append(fn())
    finally:
        dev.call("pxrhip_set_tuning", b"leaf.bin_min", old.value)
    return out


@pytest.mark.parametrize("kind", ["even", "bunch", "hot"])
@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("n", [65537, 524287, 524288])
def test_depositions(dev, grid, n, kind):
    rng = np.random.default_rng(n + grid[0])
    shape = tuple(g + 1 + 2 * NG for g in grid)
    u = [rng.uniform(-1.0, 1.0, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    P = [T(dev, a) for a in (*positions(rng, n, grid, kind), *u, g, rng.uniform(0.5, 2.0, n))]
    geo = (0.0, 0.0, 0.0)

    def current(algo):
        J = [TG(dev, np.zeros(shape)) for _ in range(3)]
        dev.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in P], -1.1, *geo,
                 0.3, 1.0, 1.0, 1.0, *grid, NG, NG, NG, 1, 1, 1, algo, 0)
        return [HG(j) for j in J]

    def rho():
        r = TG(dev, np.zeros(shape))
        dev.call("pxrhip_depose_rho_n", r.ptr, n, *[P[k].ptr for k in (0, 1, 2, 7)], -1.1, *geo,
                 1.0, 1.0, 1.0, *grid, NG, NG, NG, 2, 2, 2, 1, 0)
        return [HG(r)]

    for fn in (lambda: current(0), lambda: current(3), rho):
        for a, b in zip(*both(dev, fn)):
            assert np.abs(a).max() > 0
            assert np.abs(a - b).max() <= n * np.finfo(float).eps * np.abs(a).max()


@pytest.mark.parametrize("kind", ["even", "bunch", "hot"])
@pytest.mark.parametrize("grid", GRIDS[2:])
def test_gather(dev, grid, kind):
    """an output is a sum of at most 4^3 field values with weights that add up
    to one: 70 roundings of the largest"""
    n = 1000003
    rng = np.random.default_rng(grid[0])
    shape = tuple(g + 1 + 2 * NG for g in grid)
    P = [T(dev, a) for a in positions(rng, n, grid, kind)]
    F = [TG(dev, rng.standard_normal(shape)) for _ in range(6)]

    def gather():
        e = [T(dev, np.zeros(n)) for _ in range(6)]
        dev.call("pxrhip_geteb3d_energy_conserving", n, *[a.ptr for a in P], *[a.ptr for a in e],
                 0.0, 0.0, 0.0, 1.0, 1.0, 1.0, *grid, NG, NG, NG, 3, 3, 3, *[f.ptr for f in F], 0,
                 1, 8, 0, 0)
        return [H(a) for a in e]

    top = max(np.abs(HG(f)).max() for f in F)
    for a, b in zip(*both(dev, gather)):
        assert np.abs(a).max() > 0
        assert np.abs(a - b).max() <= 70 * np.finfo(float).eps * top
