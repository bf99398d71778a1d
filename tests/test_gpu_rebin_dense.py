"""The ordering pass of the re-binning on bins of every size class: up to 16
and 32 particles (exchange networks), up to 1024 (a wave counts ranks),
beyond (a wave's radix sort).  The output is numpy's stable argsort by bin,
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from picsar_amd import _lib
    _lib.call("pxrhip_init", 0)


@pytest.mark.parametrize("counts", [(1, 2, 15, 16), (17, 31, 32, 33), (63, 64, 65, 1000),
                                    (1023, 1024, 1025, 5000), (40000,)])
def test_bins_keep_source_order(dev, counts):
    from picsar_amd.sim import Simulation
    rng = np.random.default_rng(len(counts) + counts[0])
    sim = Simulation(8, 8, 8, order=1)
    # cell c of the x row holds counts[c] particles, in random source order;
    # the tile's sorting cells are offset by half a cell
    cell = rng.permutation(np.repeat(np.arange(len(counts)), counts))
    n = len(cell)
    x = cell + 0.75 + 0.5 * rng.random(n)
    y, z = 2.75 + 0.5 * rng.random(n), 3.75 + 0.5 * rng.random(n)
    w = 1.0 + np.arange(n)
    sp = sim.add_species("e", -1.0, 1.0, x, y, z, *np.zeros((3, n)), w)
    o = np.argsort(cell, kind="stable")
    a = sp.arrays()
    np.testing.assert_array_equal(a["w"], w[o])
    np.testing.assert_array_equal(a["x"], x[o])
