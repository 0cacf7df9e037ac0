"""Dam-break targets are shared between four lanes up to 98,304 rows.  On both
sides of that line, and at the smallest sizes, the passes agree with the plain
walk to the rounding of sums in another order, and with and without in-range
masks bit for bit."""
import numpy as np
import pytest

from cmag_amd import _lib as L
from cmag_amd import scenarios as S
from cmag_amd.systems import ParamSystem

pytestmark = pytest.mark.gpu


def stepped(sc, walk, masks, steps=1):
    vel = np.zeros_like(sc.pos)
    fl = sc.pos[:, 3] == 4.0
    vel[fl, :3] = np.random.default_rng(2).normal(scale=0.2, size=(int(fl.sum()), 3))
    s = ParamSystem.from_state(sc.params, sc.pos, vel)
    s.set_subcell_walk(walk)
    if walk:
        s.set_inrange_masks(masks)
    for _ in range(steps):
        s.update()
    return [np.asarray(s.getArray(a), np.float64) for a in (L.ARRAY_MEASURES, L.ARRAY_ACCELERATION)]


@pytest.mark.parametrize("cells,rows", [(2, None), (7, None), (24, False), (28, True)])
@pytest.mark.parametrize("order,xbits", [(L.HASH_LINEAR, 0), (L.HASH_MORTON, 4)])
def test_density_and_force(device, cells, rows, order, xbits):
    sc = S.dambreak3d(dx=0.4 / cells, hash_order=order, morton_xbits=xbits)
    if rows is not None:
        assert (sc.pos.shape[0] > 98304) == rows
    m, a = stepped(sc, True, True)
    m1, a1 = stepped(sc, True, False)
    mp, ap = stepped(sc, False, False)
    assert np.array_equal(m, m1) and np.array_equal(a, a1)
    # sums of up to 150 positive terms, each way within 150 / 2 rounding errors:
    # 75 * 6e-8 = 4.5e-6; forces cancel, normwise ten times that
    assert np.max(np.abs(m[:, 0] - mp[:, 0]) / mp[:, 0]) <= 4.5e-6
    assert np.linalg.norm(a - ap) <= 4.5e-5 * np.linalg.norm(ap)
