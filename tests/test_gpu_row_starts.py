"""Rows of a plane whose starts are staged by one lane of a unit's sixteen and
read by another: row counts around the sixteen lanes and the 96 staged rows,
with empty rows among full ones.

As in test_gpu_work_items: the charge density of the work items against the
leaf routine on the same particles, where a particle left out or taken twice
changes it by a particle's charge; the bar is n roundings of the largest node
value.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [48, 1024])
@pytest.mark.parametrize("ny", [1, 2, 15, 16, 17, 31, 32, 33, 95, 96, 97, 112, 113])
def test_rows_by_other_lanes(ny, chunk):
    from picsar_amd import _lib
    from picsar_amd.devmem import DeviceArray, DeviceGrid
    from picsar_amd.sim import Simulation
    _lib.call("pxrhip_init", 0)
    old = C.c_int64()
    _lib.call("pxrhip_get_tuning", b"fused.chunk", C.byref(old))
    n = (4, max(ny, 4), 5)
    rng = np.random.default_rng(ny)
    rows = np.flatnonzero(rng.random(ny) < 0.6) if ny > 2 else np.arange(ny)
    npart = 60 * len(rows)
    sim = Simulation(*n, 1.0, 1.0, 1.0, 0.0, 0.0, 0.0, 1, 1, 1, order=1)
    pos = [4 * rng.random(npart), rng.choice(rows, npart) + rng.random(npart),
           5 * rng.random(npart)]
    sim.add_species("e", -1.0, 1.0, *pos, *np.zeros((3, npart)), 0.5 + rng.random(npart))
    sp, g = sim.species[0], sim.ng
    want, got = DeviceGrid(*n, g), DeviceGrid(*n, g)
    a = sp.arrays()
    d = [DeviceArray.from_numpy(np.ascontiguousarray(a[k], dtype=np.float64))
         for k in ("x", "y", "z", "w")]
    _lib.call("pxrhip_depose_rho_n", want.ptr, npart, *(v.ptr for v in d), sp.q, sim.xmin,
              sim.ymin, sim.zmin, sim.dx, sim.dy, sim.dz, *n, g, g, g, 1, 1, 1, 1, 0)
    s = sp.struct(sp.cur)
    _lib.call("pxrhip_set_tuning", b"fused.chunk", chunk)
    try:
        _lib.call("pxrhip_tiles_depose_rho", C.byref(sim.grid), C.byref(s), got.ptr, 1)
        _lib.call("pxrhip_tiles_check")
    finally:
        _lib.call("pxrhip_set_tuning", b"fused.chunk", old.value)
    want, got = want.numpy(), got.numpy()
    assert np.abs(want).max() > 0
    assert np.abs(got - want).max() <= (npart + 8) * np.finfo(float).eps * np.abs(want).max()


@pytest.mark.parametrize("chunk", [16, 40, 4096])
@pytest.mark.parametrize("dense", [0.0, 0.1, 1.0])
def test_many_units(dense, chunk):
    """more units (planes of tiles) than are each given to sixteen lanes:
    neighbouring ones with rows to cut, heads and members of groups, and empty
    ones, in every mixture"""
    from picsar_amd import _lib
    from picsar_amd.devmem import DeviceArray, DeviceGrid
    from picsar_amd.sim import Simulation
    _lib.call("pxrhip_init", 0)
    old = C.c_int64()
    _lib.call("pxrhip_get_tuning", b"fused.chunk", C.byref(old))
    n, tiles = (64, 64, 64), (16, 16, 16)  # 4096 tiles of four planes and more
    rng = np.random.default_rng(int(10 * dense) + chunk)
    npart = 400000
    pos = [64 * rng.random(npart) for _ in n]
    pos[2][:100000] = np.floor(pos[2][:100000]) % 8 + rng.random(100000)  # dense planes below
    keep = rng.random(4096) < (0.3 if dense == 0.0 else 0.7)  # tiles left empty
    tile = [np.floor(a / 4).astype(int) for a in pos]
    k = keep[tile[0] + 16 * (tile[1] + 16 * tile[2])] | (rng.random(npart) < dense)
    pos = [a[k] for a in pos]
    npart = len(pos[0])
    sim = Simulation(*n, 1.0, 1.0, 1.0, 0.0, 0.0, 0.0, *tiles, order=1)
    sim.add_species("e", -1.0, 1.0, *pos, *np.zeros((3, npart)), 0.5 + rng.random(npart))
    sp, g = sim.species[0], sim.ng
    want, got = DeviceGrid(*n, g), DeviceGrid(*n, g)
    a = sp.arrays()
    d = [DeviceArray.from_numpy(np.ascontiguousarray(a[k], dtype=np.float64))
         for k in ("x", "y", "z", "w")]
    _lib.call("pxrhip_depose_rho_n", want.ptr, npart, *(v.ptr for v in d), sp.q, sim.xmin,
              sim.ymin, sim.zmin, sim.dx, sim.dy, sim.dz, *n, g, g, g, 1, 1, 1, 1, 0)
    s = sp.struct(sp.cur)
    _lib.call("pxrhip_set_tuning", b"fused.chunk", chunk)
    try:
        _lib.call("pxrhip_tiles_depose_rho", C.byref(sim.grid), C.byref(s), got.ptr, 1)
        _lib.call("pxrhip_tiles_check")
    finally:
        _lib.call("pxrhip_set_tuning", b"fused.chunk", old.value)
    want, got = want.numpy(), got.numpy()
    assert np.abs(got - want).max() <= (npart + 8) * np.finfo(float).eps * np.abs(want).max()
