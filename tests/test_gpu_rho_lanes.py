"""pxrhip_tiles_depose_rho on work items of every remainder: a thread takes
its particles in pairs, up to 16 at a time (4 at order 1, 8 at order 2).

Against pxr_depose_rho_n on the same particles.  At most n terms of one sign
are added at a node, in either order, so the bar is n roundings of the
largest node value.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 511, 513, 1025, 2047, 4095, 4097, 9001])
def test_remainders(n, order, precision):
    from picsar_amd import _lib
    from picsar_amd.devmem import DeviceArray, DeviceGrid
    from picsar_amd.sim import Simulation
    rng = np.random.default_rng(n + order)
    sim = Simulation(9, 10, 7, order=order, precision=precision)
    pos = [rng.random(n) * m for m in (9, 10, 7)]
    sim.add_species("e", -1.0, 1.0, *pos, *np.zeros((3, n)), 0.5 + rng.random(n))
    sp, g = sim.species[0], sim.ng
    want, got = DeviceGrid(9, 10, 7, g), DeviceGrid(9, 10, 7, g)
    a = sp.arrays()
    d = [DeviceArray.from_numpy(np.ascontiguousarray(a[k], dtype=np.float64))
         for k in ("x", "y", "z", "w")]
    _lib.call("pxrhip_depose_rho_n", want.ptr, n, *(v.ptr for v in d), sp.q, sim.xmin, sim.ymin,
              sim.zmin, sim.dx, sim.dy, sim.dz, 9, 10, 7, g, g, g, order, order, order, 1, 0)
    s = sp.struct(sp.cur)
    _lib.call("pxrhip_tiles_depose_rho", C.byref(sim.grid), C.byref(s), got.ptr, order)
    _lib.call("pxrhip_tiles_check")
    want, got = want.numpy(), got.numpy()
    assert np.abs(want).max() > 0
    assert np.abs(got - want).max() <= (n + 8) * np.finfo(float).eps * np.abs(want).max()
