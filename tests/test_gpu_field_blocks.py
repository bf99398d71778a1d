"""Field updates whose blocks fill the rounds of the XCDs partly, just and
just not (a round of the Yee updates is 256 blocks of 256 nodes, one of the
order-4 march 128 blocks of 64 x 4 columns): every node once, bit for bit as
the oracle has it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

G = 2


@pytest.mark.parametrize("n", [(4, 4, 4), (255, 15, 15), (255, 15, 16), (256, 15, 15),
                               (63, 63, 15), (64, 40, 33), (127, 127, 9), (61, 45, 70)])
@pytest.mark.parametrize("norder", [2, 4])
def test_every_node_once(orc, n, norder):
    from picsar_amd import _lib
    from picsar_amd.picsarpy import picsar as pxr
    from picsar_amd.sim import _fd_weights
    _lib.call("pxrhip_init", 0)
    rng = np.random.default_rng(sum(n))
    A = [np.asfortranarray(rng.standard_normal([m + 1 + 2 * G for m in n])) for _ in range(9)]
    lo, hi, alo, ahi = (0, 0, 0), n, (-G,) * 3, tuple(m + G for m in n)
    s, g = (0.31, 0.27, 0.36), (G,) * 3
    we, wb, ge, gb = ([x.copy(order="F") for x in A] for _ in range(4))
    if norder == 2:
        orc.push_em3d_evec(lo, hi, *we, 0.3, *s, *n, *g)
        orc.push_em3d_bvec(lo, hi, *wb[:6], *s, *n, *g)
        pxr.pxrpush_em3d_evec(*(lo, hi) * 3, *sum(([f, alo, ahi] for f in ge), []), 0.3, *s)
        pxr.pxrpush_em3d_bvec(*(lo, hi) * 3, *sum(([f, alo, ahi] for f in gb[:6]), []), *s)
    else:
        c = [v * _fd_weights(4) for v in s]
        orc.push_em3d_evec_norder(*we, 0.3, *c, *n, 4, 4, 4, *g, 0, 0, 0, l_nodal=False)
        orc.push_em3d_bvec_norder(*wb[:6], *c, *n, 4, 4, 4, *g, 0, 0, 0, l_nodal=False)
        pxr.pxrpush_em3d_evec_norder(*ge, 0.3, *c, *n, 4, 4, 4, *g, 0, 0, 0, False)
        pxr.pxrpush_em3d_bvec_norder(*gb[:6], *c, *n, 4, 4, 4, *g, 0, 0, 0, False)
    for a, b in zip(ge[:3] + gb[3:6], we[:3] + wb[3:6]):
        np.testing.assert_array_equal(a, b)
