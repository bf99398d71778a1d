"""Large leaf calls where the library's scratch is limited (scratch.limit):
the order of the particles comes before the optional records, a gather takes
smaller parts, the sort stages one array at a time, and a call without memory
for any of it takes the unbinned kernels.  Buffers beyond 1 GiB are given back.

Currents against the same call without a limit: a node's sum has at most n
terms in another order, n roundings of the largest node.  The gather has the bar
of test_gpu_leafgather, the sort is bit for bit.
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, SHAPE, H, HG, T, TG, particles

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


@pytest.fixture
def limit(dev):
    def set_limit(n):
        dev.call("pxrhip_set_tuning", b"scratch.limit", int(n))
        assert get(dev, b"scratch.bytes") == 0
    yield set_limit
    set_limit(0)


def get(dev, key):
    v = C.c_int64()
    dev.call("pxrhip_get_tuning", key, C.byref(v))
    return v.value


def plasma(dev, n):
    rng = np.random.default_rng(n)
    u = [rng.uniform(-1.0, 1.0, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    return [T(dev, a) for a in (*particles(rng, n, margin=1.0), *u, g, rng.uniform(0.5, 2.0, n))]


# 600,000 particles: 9.6 MB for their order, a little for blocks and items,
# 38.4 MB of records
@pytest.mark.parametrize("algo", [0, 3])
@pytest.mark.parametrize("mb,form,records", [(64, 1, 1), (44, 1, 0), (20, 1, 0), (8, 0, 0)])
def test_current(dev, limit, mb, form, records, algo):
    n = 600000
    P = plasma(dev, n)

    def run():
        J = [TG(dev, np.zeros(SHAPE)) for _ in range(3)]
        dev.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in P], -1.1, 0.0,
                 0.0, 0.0, 0.3, 1.0, 1.0, 1.0, NX, NY, NZ, NG, NG, NG, 1, 1, 1, algo, 0)
        return [HG(j) for j in J]

    limit(0)
    want = run()
    assert (get(dev, b"last.leaf_current"), get(dev, b"last.leaf_records")) == (1, 1)
    limit(mb * MB)
    for _ in range(2):  # also with what the first call has left
        got = run()
        assert (get(dev, b"last.leaf_current"), get(dev, b"last.leaf_records")) == (form, records)
        assert get(dev, b"scratch.bytes") <= mb * MB
        for a, b in zip(want, got):
            assert np.abs(a - b).max() <= n * np.finfo(float).eps * np.abs(a).max()


def test_records_of_an_earlier_call_make_room(dev, limit):
    """a larger order 3 call, which has no records, takes their memory"""
    limit(64 * MB)
    for n, order, records in ((600000, 1, 1), (2000000, 3, 0)):
        P = plasma(dev, n)
        J = [TG(dev, np.zeros(SHAPE)) for _ in range(3)]
        dev.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in P], -1.1, 0.0,
                 0.0, 0.0, 0.3, 1.0, 1.0, 1.0, NX, NY, NZ, NG, NG, NG, order, order, order, 0, 0)
        assert (get(dev, b"last.leaf_current"), get(dev, b"last.leaf_records")) == (1, records)


@pytest.mark.parametrize("mb,form", [(0, 1), (64, 1), (30, 0)])
def test_gather(dev, limit, mb, form):
    """1.6 million: 25.6 MB for their order, 76.8 of records (64 MB: in parts)"""
    n, grid, ng = 1600000, (80, 80, 80), 2
    rng = np.random.default_rng(5)
    P = [T(dev, rng.uniform(1.0, g - 1.0, n)) for g in grid]
    F = [rng.standard_normal(tuple(g + 1 + 2 * ng for g in grid)) for _ in range(6)]
    FD = [TG(dev, f) for f in F]
    out = []
    for m, want in ((0, 1), (mb, form)):
        limit(m * MB)
        e = [T(dev, np.zeros(n)) for _ in range(6)]
        dev.call("pxrhip_geteb3d_energy_conserving", n, *[a.ptr for a in P], *[a.ptr for a in e],
                 0.0, 0.0, 0.0, 1.0, 1.0, 1.0, *grid, ng, ng, ng, 3, 3, 3, *[f.ptr for f in FD], 0,
                 1, 8, 0, 0)
        assert get(dev, b"last.leaf_gather") == want
        out.append([H(a) for a in e])
    for f, a, b in zip(F, *out):
        assert np.abs(a - b).max() <= 70 * np.finfo(float).eps * np.abs(f).max()


def test_rho_and_sort(dev, limit):
    n = 200003
    P = plasma(dev, n)
    rng = np.random.default_rng(6)
    S = [rng.uniform(0, c, n) for c in (23, 17, 11)] + [rng.standard_normal(n) for _ in range(5)]
    o = np.argsort((np.floor(S[2]) * 17 + np.floor(S[1])) * 23 + np.floor(S[0]), kind="stable")
    rho = []
    # 16 MB: sorts with all arrays staged at once; 5: one at a time; 2: fails
    for mb, sorts in ((0, True), (16, True), (5, True), (2, False)):
        limit(mb * MB)
        D = [T(dev, a) for a in S]
        args = (n, *[d.ptr for d in D], 1, 0.0, 0.0, 0.0, 23.0, 17.0, 11.0, 1.0, 1.0, 1.0)
        if sorts:
            dev.call("pxrhip_particle_bin_sorting", *args)
        else:
            with pytest.raises(dev.PxrHipError, match="scratch"):
                dev.call("pxrhip_particle_bin_sorting", *args)
        for d, a in zip(D, S):
            np.testing.assert_array_equal(H(d), a[o] if sorts else a)
        limit(mb * MB)
        r = TG(dev, np.zeros(SHAPE))
        dev.call("pxrhip_depose_rho_n", r.ptr, n, *[P[k].ptr for k in (0, 1, 2, 7)], -1.1, 0.0,
                 0.0, 0.0, 1.0, 1.0, 1.0, NX, NY, NZ, NG, NG, NG, 2, 2, 2, 1, 0)
        assert get(dev, b"last.leaf_rho") == (mb != 2)
        rho.append(HG(r))
    for r in rho[1:]:
        assert np.abs(r - rho[0]).max() <= n * np.finfo(float).eps * np.abs(rho[0]).max()


def test_large_buffers_are_given_back(dev, limit):
    """18 million particles on 270^3 cells: one part, 1.15 GB of records"""
    n, grid = 18000000, (270, 270, 270)
    rng = np.random.default_rng(7)
    x = [T(dev, rng.uniform(1.0, g - 1.0, n)) for g in grid]
    one = T(dev, np.ones(n))
    zero = T(dev, np.zeros(n))
    J = [TG(dev, np.zeros(tuple(g + 1 + 2 * NG for g in grid))) for _ in range(3)]
    limit(0)
    for checks, records in ((1, 1), (0, 0)):
        dev.call("pxrhip_set_checks", checks)
        try:
            dev.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in x],
                     *[zero.ptr] * 3, one.ptr, one.ptr, -1.1, 0.0, 0.0, 0.0, 0.3, 1.0, 1.0, 1.0,
                     *grid, NG, NG, NG, 1, 1, 1, 0, 0)
        finally:
            dev.call("pxrhip_set_checks", 1)
        assert (get(dev, b"last.leaf_current"), get(dev, b"last.leaf_records")) == (1, records)
        dev.call("pxrhip_synchronize")
        assert get(dev, b"scratch.bytes") < 1 << 30
