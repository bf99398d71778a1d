"""The unbinned deposition of the leaf routines at the ends of a wave, of a
block of waves (64 * 16 particles) and of the chip (256 per CU), where every
particle has to be taken once.

Against the oracle; a node's sum has at most n terms of one order of
magnitude, so the bar is n roundings relative to the largest value.
"""
import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, HG, T, TG, SHAPE, particles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


@pytest.mark.parametrize("algo", [0, 3])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 65535, 65537])
def test_every_particle_once(dev, n, algo):
    """total current = sum of q w v over the particles, whatever the order"""
    from picsar_amd.picsarpy import picsar
    from picsar_amd import _lib
    import ctypes
    rng = np.random.default_rng(n)
    x, y, z = particles(rng, n, margin=1.0)
    u = [rng.uniform(0.1, 0.3, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    w = rng.uniform(0.5, 2.0, n)
    J = [TG(dev, np.zeros(SHAPE)) for _ in range(3)]
    old = ctypes.c_int64()
    _lib.call("pxrhip_get_tuning", b"leaf.bin_min", ctypes.byref(old))
    _lib.call("pxrhip_set_tuning", b"leaf.bin_min", 0)
    was, picsar.l_nodalgrid = picsar.l_nodalgrid, False
    try:
        P = [T(dev, a) for a in (x, y, z, *u, g, w)]
        picsar.depose_jxjyjz(*J, n, *P, -1.1, 0.0, 0.0, 0.0, 0.45, 1.0, 1.0, 1.0, NX, NY, NZ,
                             NG, NG, NG, 2, 2, 2, algo)
    finally:
        _lib.call("pxrhip_set_tuning", b"leaf.bin_min", old.value)
        picsar.l_nodalgrid = was
    for j, c in zip(J, u):
        want = -1.1 * np.sum(w * c * g)
        assert abs(HG(j).sum() - want) <= (n + 200) * 8 * np.finfo(float).eps * abs(want)


@pytest.mark.parametrize("algo", [0, 3])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("n,ordered", [(524287, False), (524288, False), (524288, True),
                                       (8388609, False)])
def test_binned_sets_with_and_without_records(dev, n, ordered, order, algo):
    """A set in no order is deposited from records of its particles (orders 1
    and 2), beyond eight million in parts; against the unbinned form, whose
    sums differ in their order alone."""
    from picsar_amd.picsarpy import picsar
    from picsar_amd import _lib
    import ctypes
    rng = np.random.default_rng(n + order)
    x, y, z = particles(rng, n, margin=1.0)
    if ordered:
        o = np.lexsort((np.floor(x), np.floor(y), np.floor(z)))
        x, y, z = x[o], y[o], z[o]
    x[n // 2] = 1e3  # skipped by both
    u = [rng.uniform(-1.0, 1.0, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    P = [T(dev, a) for a in (x, y, z, *u, g, rng.uniform(0.5, 2.0, n))]
    old = ctypes.c_int64()
    _lib.call("pxrhip_get_tuning", b"leaf.bin_min", ctypes.byref(old))
    was, picsar.l_nodalgrid = picsar.l_nodalgrid, False
    res = []
    try:
        for bin_min in (0, 1):
            _lib.call("pxrhip_set_tuning", b"leaf.bin_min", bin_min)
            J = [TG(dev, np.zeros(SHAPE)) for _ in range(3)]
            with pytest.raises(_lib.PxrHipError, match="1 particle"):
                picsar.depose_jxjyjz(*J, n, *P, -1.1, 0.0, 0.0, 0.0, 0.3, 1.0, 1.0, 1.0, NX, NY,
                                     NZ, NG, NG, NG, order, order, order, algo)
            res.append([HG(j) for j in J])
    finally:
        _lib.call("pxrhip_set_tuning", b"leaf.bin_min", old.value)
        picsar.l_nodalgrid = was
    # a node's sum of at most n/100 terms of up to 2.2 |q w v| each, either order
    tol = n / 100 * np.finfo(float).eps * 2.2 * (n / 100)
    for a, b in zip(*res):
        assert np.abs(a).max() > 0
        assert np.abs(a - b).max() <= tol
