"""The order-3 Esirkepov step of an FP64 species of one or two particles per
cell, whose lanes are not dealt by LDS bank, against the oracle at the step's
bar (1e-12 relative in norm: the order of the sums differs), for every gather
and pusher; and which form is taken by the species' capacity per cell.
"""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_step import build, rel

pytestmark = pytest.mark.gpu


def banks():
    from picsar_amd import _lib
    v = C.c_int64()
    _lib.call("pxrhip_get_tuning", b"last.bank_lanes", C.byref(v))
    return v.value


@pytest.mark.parametrize("lo,pusher", [(True, "vay"), (True, "boris"), (False, "vay"),
                                       (False, "boris")])
@pytest.mark.parametrize("ppc,form", [(1, 0), (2, 0), (3, 1)])
def test_step(orc, ppc, form, lo, pusher):
    from picsar_amd import _lib
    _lib.call("pxrhip_init", 0)
    sim, ref, tng = build(None, orc, 3, lo, pusher, "esirkepov", ppc=ppc)
    sim.step(2)
    assert banks() == form
    ref.step()
    ref.step()
    for k in ("ex", "ey", "ez", "bx", "by", "bz", "jx", "jy", "jz"):
        assert rel(tng(sim.fields[k]), ref.f[k]) <= 1e-12, k


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("capacity,form", [(767, 1), (768, 0), (2559, 0), (2560, 1)])
def test_rule(capacity, form, precision):
    """1024 cells: from three in four up to two and a half, FP64 only"""
    from picsar_amd import _lib
    from picsar_amd.sim import Simulation
    _lib.call("pxrhip_init", 0)
    sim = Simulation(16, 8, 8, 1.0, 1.0, 1.0, 0.0, 0.0, 0.0, 2, 1, 1, order=3, precision=precision)
    rng = np.random.default_rng(1)
    x = [rng.uniform(0, m, 500) for m in (16, 8, 8)]
    sim.add_species("e", -1.0, 1.0, *x, *np.zeros((3, 500)), np.ones(500), capacity=capacity)
    sim.step(1)
    assert banks() == (form if precision == "fp64" else 1)
