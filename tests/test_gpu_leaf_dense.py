"""Leaf depositions of order 3 of dense sets in cell order, where the lanes of
a wave spread over the whole work item: item sizes around a workgroup, cells of
few and of many particles, sets whose order ends halfway.

Against the unbinned form on the same particles: a node's sum has at most n
terms, added in another order, so the bar is n roundings of the largest node.
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, SHAPE, HG, T, TG

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


@pytest.mark.parametrize("order_of", ["cells", "half", "one cell"])
@pytest.mark.parametrize("n,cells", [(700, 4), (1025, 8), (70001, 12), (70001, 3), (262147, 12)])
@pytest.mark.parametrize("chunk", [255, 257, 300, 1000, 4096])
def test_dense_sets(dev, n, cells, chunk, order_of):
    rng = np.random.default_rng(n + cells)
    x = [rng.uniform(1.0, 1.0 + (1 if order_of == "one cell" else cells), n) for _ in range(3)]
    o = np.lexsort(tuple(np.floor(a) for a in x))
    if order_of == "half":
        rng.shuffle(o[n // 2:])
    x = [a[o] for a in x]
    u = [rng.uniform(-1.0, 1.0, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    P = [T(dev, a) for a in (*x, *u, g, rng.uniform(0.5, 2.0, n))]
    geo = (-1.1, 0.0, 0.0, 0.0)

    def run():
        res = []
        for algo in (0, 3):
            J = [TG(dev, np.zeros(SHAPE)) for _ in range(3)]
            dev.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in P], *geo, 0.3,
                     1.0, 1.0, 1.0, NX, NY, NZ, NG, NG, NG, 3, 3, 3, algo, 0)
            res += [HG(j) for j in J]
        r = TG(dev, np.zeros(SHAPE))
        dev.call("pxrhip_depose_rho_n", r.ptr, n, *[P[k].ptr for k in (0, 1, 2, 7)], *geo, 1.0, 1.0,
                 1.0, NX, NY, NZ, NG, NG, NG, 3, 3, 3, 1, 0)
        return res + [HG(r)]

    old = {k: C.c_int64() for k in (b"leaf.bin_min", b"leaf.bin_chunk")}
    for k, v in old.items():
        dev.call("pxrhip_get_tuning", k, C.byref(v))
    try:
        dev.call("pxrhip_set_tuning", b"leaf.bin_chunk", chunk)
        out = []
        for bin_min in (0, 1):
            dev.call("pxrhip_set_tuning", b"leaf.bin_min", bin_min)
            out.append(run())
        form = C.c_int64()
        dev.call("pxrhip_get_tuning", b"last.leaf_rho", C.byref(form))
        assert form.value == 1
    finally:
        for k, v in old.items():
            dev.call("pxrhip_set_tuning", k, v.value)
    for a, b in zip(*out):
        assert np.abs(a).max() > 0
        assert np.abs(a - b).max() <= n * np.finfo(float).eps * np.abs(a).max()
