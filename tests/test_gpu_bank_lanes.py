"""Order-3 Esirkepov deposition with lanes dealt by LDS bank (bank_slots in
pxr_fused.h): the particles of a work item in sixteen classes, classes with
more than their share filling the lanes that others leave empty.

Particle sets that fill the classes unevenly (all in one cell, in one row of
cells, fewer than a wave, a few more than a wave or a round) against the FP64
oracle: the step's bar, 1e-12 relative in norm, since only the order in which
contributions meet changes.  Every gather and pusher variant of the order is
run, as each is a kernel of its own; mixed precision at its bar of 1e-5."""
import numpy as np
import pytest

from tests.test_gpu_step import build, rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    from picsar_amd import _lib
    _lib.call("pxrhip_init", 0)
    return None


def add_both(sim, ref, rng, n, lo, hi):
    """n particles in the box lo..hi (cells), in the simulation and the oracle."""
    x = [rng.uniform(a, b, n) * d + o for a, b, d, o in zip(
        lo, hi, (sim.dx, sim.dy, sim.dz), (sim.xmin, sim.ymin, sim.zmin))]
    u = [rng.standard_normal(n) * 0.3 for _ in range(3)]
    w = (1.0 + np.arange(n)) / n * 2.0 ** -10
    w = w.astype(np.float32).astype(np.float64)
    u = [a.astype(np.float32).astype(np.float64) for a in u]
    ref.add_species(-1.0, 1.0, *x, *u, w)
    sim.add_species("more", -1.0, 1.0, *x, *u, w, gaminv=ref.species[-1]["gaminv"])


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("lo,pusher", [(True, "vay"), (True, "boris"), (False, "vay"),
                                       (False, "boris")])
def test_kernel_variants(torch, orc, precision, tol, lo, pusher):
    kw = {} if precision == "fp64" else dict(precision="mixed", id_scale=2.0 ** -15, ppc=2)
    sim, ref, tng = build(torch, orc, 3, lo, pusher, "esirkepov", **kw)
    add_both(sim, ref, np.random.default_rng(1), 700, (3, 3, 3), (7, 6, 5))
    sim.step(1)
    ref.step()
    for k in ("ex", "ey", "ez", "bx", "by", "bz", "jx", "jy", "jz"):
        assert rel(tng(sim.fields[k]), ref.f[k]) <= tol, k


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 257, 4096, 5001])
@pytest.mark.parametrize("box", [((4.0, 4.0, 4.0), (4.4, 4.4, 4.4)),    # one cell, one class
                                 ((1.0, 4.0, 4.0), (7.0, 4.4, 4.4)),    # a row of cells
                                 ((1.0, 1.0, 1.0), (7.0, 7.0, 7.0))])
def test_uneven_classes(torch, orc, n, box):
    sim, ref, tng = build(torch, orc, 3, True, "vay", "esirkepov", seed=3)
    add_both(sim, ref, np.random.default_rng(n), n, *box)
    sim.step(1)
    ref.step()
    for k in ("ex", "ey", "ez", "jx", "jy", "jz"):
        assert rel(tng(sim.fields[k]), ref.f[k]) <= 1e-12, k


def test_large_chunk(torch, orc):
    """A work-item size beyond the 16-bit slots is taken as a smaller one."""
    sim, ref, tng = build(torch, orc, 3, True, "vay", "esirkepov", chunk=1 << 20, ntiles=(1, 1, 1))
    add_both(sim, ref, np.random.default_rng(8), 70000, (4.0, 4.0, 4.0), (4.4, 4.4, 4.4))
    sim.step(1)
    ref.step()
    for k in ("ex", "ey", "ez", "jx", "jy", "jz"):
        assert rel(tng(sim.fields[k]), ref.f[k]) <= 1e-12, k
