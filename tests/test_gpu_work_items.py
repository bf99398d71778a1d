"""Work items of tiles with more rows than are staged at once (96), of planes
cut into more items than are kept from the counting pass (16), of rows denser
than an item, and of many units.

The charge density of the work items against the leaf routine on the same
particles: one left out or taken twice changes it by a particle's charge.
The bar is n roundings of the largest node value.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [64, 4096])
@pytest.mark.parametrize("n,tiles,npart", [((5, 130, 4), (1, 1, 1), 20000),
                                           ((4, 95, 3), (1, 1, 1), 3000),
                                           ((4, 96, 3), (1, 1, 1), 900),
                                           ((6, 17, 40), (1, 1, 1), 12000),
                                           ((64, 65, 66), (16, 16, 16), 60000)])
def test_every_particle_in_one_item(n, tiles, npart, chunk):
    from picsar_amd import _lib
    from picsar_amd.devmem import DeviceArray, DeviceGrid
    from picsar_amd.sim import Simulation
    old = C.c_int64()
    _lib.call("pxrhip_init", 0)
    _lib.call("pxrhip_get_tuning", b"fused.chunk", C.byref(old))
    rng = np.random.default_rng(npart)
    sim = Simulation(*n, 1.0, 1.0, 1.0, 0.0, 0.0, 0.0, *tiles, order=2)
    pos = [rng.random(npart) * m for m in n]
    pos[1][: npart // 4] = 2.5 + 0.1 * rng.random(npart // 4)  # dense rows
    pos[2][: npart // 8] = 1.5 + 0.1 * rng.random(npart // 8)
    pos[1][npart // 2: npart // 2 + npart // 4] *= 0.3  # empty rows and planes elsewhere
    sim.add_species("e", -1.0, 1.0, *pos, *np.zeros((3, npart)), 0.5 + rng.random(npart))
    sp, g = sim.species[0], sim.ng
    want, got = DeviceGrid(*n, g), DeviceGrid(*n, g)
    a = sp.arrays()
    d = [DeviceArray.from_numpy(np.ascontiguousarray(a[k], dtype=np.float64))
         for k in ("x", "y", "z", "w")]
    _lib.call("pxrhip_depose_rho_n", want.ptr, npart, *(v.ptr for v in d), sp.q, sim.xmin,
              sim.ymin, sim.zmin, sim.dx, sim.dy, sim.dz, *n, g, g, g, 2, 2, 2, 1, 0)
    s = sp.struct(sp.cur)
    _lib.call("pxrhip_set_tuning", b"fused.chunk", chunk)
    try:
        _lib.call("pxrhip_tiles_depose_rho", C.byref(sim.grid), C.byref(s), got.ptr, 2)
        _lib.call("pxrhip_tiles_check")
    finally:
        _lib.call("pxrhip_set_tuning", b"fused.chunk", old.value)
    want, got = want.numpy(), got.numpy()
    assert np.abs(want).max() > 0
    assert np.abs(got - want).max() <= (npart + 8) * np.finfo(float).eps * np.abs(want).max()
