"""The leaf sort beside other calls: whether it moves anything depends on its
own particles alone, not on what other calls have counted, and sorts of
several threads, which share scratch, give what they give one after the other.

Bit for bit against numpy's stable sort of the same keys.
"""
import ctypes as C
import threading

import numpy as np
import pytest

from tests.test_gpu_leaf import NG, NX, NY, NZ, SHAPE, H, T, TG, particles

pytestmark = pytest.mark.gpu

CELLS = (23, 17, 11)
BOX = (0.0, 0.0, 0.0, *map(float, CELLS), 1.0, 1.0, 1.0)


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.load()
    _lib.call("pxrhip_init", 0)
    return _lib


def sort_set(rng, n):
    P = [rng.uniform(0, c, n) for c in CELLS] + [rng.standard_normal(n) for _ in range(5)]
    key = (np.floor(P[2]) * CELLS[1] + np.floor(P[1])) * CELLS[0] + np.floor(P[0])
    o = np.argsort(key, kind="stable")
    return P, [p[o] for p in P]


def gather_with_one_outside(pxr, dev, n, F):
    x, y, z = particles(np.random.default_rng(1), n, margin=1.0)
    x[n // 2] = 1e3
    pxr.geteb3d_energy_conserving(n, *[T(dev, a) for a in (x, y, z)],
                                  *[T(dev, np.zeros(n)) for _ in range(6)], 0.0, 0.0, 0.0, 1.0,
                                  1.0, 1.0, NX, NY, NZ, NG, NG, NG, 1, 1, 1, *F, False, True)


def count(dev, reset):
    c = C.c_longlong()
    dev.call("pxrhip_bad_count", C.byref(c), reset)
    return c.value


@pytest.mark.parametrize("entry", ["pxrhip_particle_bin_sorting",
                                   "pxrhip_particle_bin_sorting_noalloc"])
def test_particles_skipped_by_an_unchecked_call(dev, entry):
    """they do not stop a later sort, and stay counted"""
    from picsar_amd.picsarpy import picsar
    rng = np.random.default_rng(3)
    P, want = sort_set(rng, 5003)
    F = [TG(dev, rng.standard_normal(SHAPE)) for _ in range(6)]
    D = [T(dev, p) for p in P]
    count(dev, 1)
    was, picsar.l_nodalgrid = picsar.l_nodalgrid, False
    dev.call("pxrhip_set_checks", 0)
    try:
        gather_with_one_outside(picsar, dev, 1000, F)
        dev.call(entry, 5003, *[d.ptr for d in D], 1, *BOX)
        assert count(dev, 1) == 1
    finally:
        dev.call("pxrhip_set_checks", 1)
        count(dev, 1)
        picsar.l_nodalgrid = was
    for d, w in zip(D, want):
        np.testing.assert_array_equal(H(d), w)


def test_sorts_of_several_threads(dev):
    """two entry points, sizes with and without a second pass of the radix
    sort, keys out of range, and a thread whose calls skip a particle"""
    from picsar_amd.picsarpy import picsar
    rng = np.random.default_rng(4)
    F = [TG(dev, rng.standard_normal(SHAPE)) for _ in range(6)]
    sets = [sort_set(rng, n) for n in (200003, 61001, 300007)]
    entries = ["pxrhip_particle_bin_sorting", "pxrhip_particle_bin_sorting_noalloc",
               "pxrhip_particle_bin_sorting"]
    rounds = 6
    D = [[[T(dev, p) for p in P] for _ in range(rounds)] for P, _ in sets]
    bad = [p.copy() for p in sets[1][0]]
    bad[0][77] = 1e6
    B = [[T(dev, p) for p in bad] for _ in range(rounds)]
    err = []

    def sorts(k):
        for r in range(rounds):
            try:
                dev.call(entries[k], len(sets[k][0][0]), *[d.ptr for d in D[k][r]], 1, *BOX)
            except Exception as e:  # noqa: BLE001 - reported by the main thread
                err.append((k, r, str(e)))

    def refused():
        for r in range(rounds):
            try:
                dev.call("pxrhip_particle_bin_sorting", 61001, *[d.ptr for d in B[r]], 1, *BOX)
                err.append(("refused", r, "was sorted"))
            except dev.PxrHipError as e:
                if "1 particle(s) have a cell key outside" not in str(e):
                    err.append(("refused", r, str(e)))

    def skips():
        for r in range(4 * rounds):
            try:
                gather_with_one_outside(picsar, dev, 1000, F)
            except dev.PxrHipError as e:
                if "skipped" not in str(e):
                    err.append(("skips", r, str(e)))

    was, picsar.l_nodalgrid = picsar.l_nodalgrid, False
    try:
        th = [threading.Thread(target=sorts, args=(k,)) for k in range(3)]
        th += [threading.Thread(target=refused), threading.Thread(target=skips)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    finally:
        picsar.l_nodalgrid = was
        count(dev, 1)
    assert not err, err
    for (_, want), rs in zip(sets, D):
        for ds in rs:
            for d, w in zip(ds, want):
                np.testing.assert_array_equal(H(d), w)
    for ds in B:
        for d, b in zip(ds, bad):
            np.testing.assert_array_equal(H(d), b)
