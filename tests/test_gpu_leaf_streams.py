"""Large leaf calls with the checks off, one after the other on two streams:
they share scratch for the order of their particles, and the second may not
touch it before the first is done.  And recorded into a graph of the caller's
own: the graph may not refer to that scratch, which a later call may free.

Each against the same call alone.  Currents and densities are sums in an order
that depends on the launch: a node's sum has at most n/100 terms of up to
2.2 |q w v| each, in either order; the gather has the bar of
test_gpu_leafgather.
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, SHAPE, HG, T, TG, particles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


@pytest.fixture
def streams(dev):
    """two streams of the library's HIP runtime; the library's own afterwards"""
    hip = C.CDLL(dev.LIB_PATH)  # its symbols include those of the runtime it is linked to
    own = dev.load().pxrhip_get_stream()
    s = [C.c_void_p(), C.c_void_p()]
    for p in s:
        assert hip.hipStreamCreate(C.byref(p)) == 0
    yield hip, s
    dev.call("pxrhip_synchronize")
    assert hip.hipDeviceSynchronize() == 0
    dev.call("pxrhip_set_stream", C.c_void_p(own))
    for p in s:
        assert hip.hipStreamDestroy(p) == 0


GEO = (0.0, 0.0, 0.0)


def current(dev, J, n, P, order, algo):
    dev.call("pxrhip_depose_jxjyjz", *[j.ptr for j in J], n, *[a.ptr for a in P], -1.1, *GEO, 0.3,
             1.0, 1.0, 1.0, NX, NY, NZ, NG, NG, NG, order, order, order, algo, 0)


def rho(dev, J, n, P, order, _):
    dev.call("pxrhip_depose_rho_n", J[0].ptr, n, *[P[k].ptr for k in (0, 1, 2, 7)], -1.1, *GEO, 1.0,
             1.0, 1.0, NX, NY, NZ, NG, NG, NG, order, order, order, 1, 0)


def plasma(dev, rng, n):
    x = particles(rng, n, margin=1.0)
    u = [rng.uniform(-1.0, 1.0, n) for _ in range(3)]
    g = 1 / np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    return [T(dev, a) for a in (*x, *u, g, rng.uniform(0.5, 2.0, n))]


@pytest.mark.parametrize("call,order,algo", [(current, 1, 3), (current, 3, 3), (current, 2, 0),
                                             (rho, 2, 0)])
def test_two_streams_in_turn(dev, streams, call, order, algo):
    _, streams = streams
    sizes = (900001, 700000, 66000, 1500007)
    rng = np.random.default_rng(order + algo)
    sets = [plasma(dev, rng, n) for n in sizes]
    alone, turn = ([[TG(dev, np.zeros(SHAPE)) for _ in range(3)] for _ in sizes] for _ in "ab")
    for J, n, P in zip(alone, sizes, sets):
        call(dev, J, n, P, order, algo)
    dev.call("pxrhip_synchronize")
    dev.call("pxrhip_set_checks", 0)
    try:
        for k, (J, n, P) in enumerate(zip(turn, sizes, sets)):
            dev.call("pxrhip_set_stream", streams[k % 2])
            call(dev, J, n, P, order, algo)
        for s in streams:
            dev.call("pxrhip_set_stream", s)
            dev.call("pxrhip_synchronize")
    finally:
        dev.call("pxrhip_set_checks", 1)
    for n, A, B in zip(sizes, alone, turn):
        tol = n / 100 * np.finfo(float).eps * 2.2 * (n / 100)
        for a, b in zip(A, B):
            assert np.abs(HG(a) - HG(b)).max() <= tol
        assert np.abs(HG(A[0])).max() > 0


@pytest.mark.parametrize("call,order,algo", [(current, 1, 3), (current, 2, 0), (rho, 1, 0)])
def test_recorded_by_the_caller(dev, streams, call, order, algo):
    """each replay adds the call's current once, also after eager calls that
    make the scratch grow"""
    hip, streams = streams
    n = 70001
    rng = np.random.default_rng(17)
    P, big = plasma(dev, rng, n), [plasma(dev, rng, m) for m in (2500003, 3500003)]
    J, once, other = ([TG(dev, np.zeros(SHAPE)) for _ in range(3)] for _ in "abc")
    dev.call("pxrhip_synchronize")
    graph, ex = C.c_void_p(), C.c_void_p()
    dev.call("pxrhip_set_checks", 0)
    try:
        dev.call("pxrhip_set_stream", streams[0])
        call(dev, once, n, P, order, algo)
        dev.call("pxrhip_synchronize")
        assert hip.hipStreamBeginCapture(streams[0], 2) == 0  # relaxed
        call(dev, J, n, P, order, algo)
        assert hip.hipStreamEndCapture(streams[0], C.byref(graph)) == 0
        assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
        for k in range(3):
            assert hip.hipGraphLaunch(ex, streams[0]) == 0
            dev.call("pxrhip_synchronize")
            if k < 2:
                call(dev, other, len(big[k][0]), big[k], order, algo)
                dev.call("pxrhip_synchronize")
    finally:
        dev.call("pxrhip_set_checks", 1)
        if ex:
            hip.hipGraphExecDestroy(ex)
        if graph:
            hip.hipGraphDestroy(graph)
    tol = 3 * n / 100 * np.finfo(float).eps * 2.2 * (3 * n / 100)
    for a, b in zip(once, J):
        assert np.abs(3 * HG(a) - HG(b)).max() <= tol
    assert np.abs(HG(once[0])).max() > 0
