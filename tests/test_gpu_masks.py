"""The walks that go through staged lookups and in-range masks equal the ones
that do not, bit for bit: every cell order visits a target's candidates in the
same order, and the orders differ in which rows and blocks take which path."""
import numpy as np
import pytest

from cmag_amd import _lib as L
from cmag_amd import scenarios as S
from cmag_amd.systems import ParamSystem

pytestmark = pytest.mark.gpu

ARRAYS = (L.ARRAY_MEASURES, L.ARRAY_ACCELERATION)


def passes(p, pos, order, xbits, vel=None):
    p = type(p).from_buffer_copy(p)
    p.hash_order, p.morton_xbits = order, xbits
    S.finalize(p)
    s = ParamSystem.from_state(p, pos, vel)
    s.update()
    out = [s.getArray(a) for a in ARRAYS]
    # measures are kept in sorted order: back to the particles'
    idx = s.getUintArray(L.ARRAY_INDEX)
    m = np.zeros_like(out[0])
    m[idx] = out[0]
    s.close()
    return m[:, :2], out[1]


# blocks of 64 targets (up to 98,304 rows four lanes share one) over one, two and
# more rows of cells, in clouds of 1 to 100 particles a cell, at the border of the
# grid and inside it
@pytest.mark.parametrize("n,rows,cells_x", [(64, 1, 3), (255, 2, 2), (257, 2, 4), (600, 3, 30), (3000, 4, 16),
                                             (2500, 5, 5)])
@pytest.mark.parametrize("border", [False, True])
def test_staged_blocks_equal_the_global_walk(device, n, rows, cells_x, border):
    sc = S.dambreak3d(dx=0.02)
    p = sc.params
    cs = [float(c) for c in p.cell_size]
    at = 0 if border else 9
    rng = np.random.default_rng(n)
    pos = np.zeros((n, 4), np.float32)
    span = (cells_x, rows, 2)
    for a in range(3):
        pos[:, a] = float(p.world_origin[a]) + cs[a] * (at + rng.uniform(0.02, span[a] - 0.02, n))
    pos[:, 3] = np.where(rng.uniform(size=n) < 0.1, 1.0, 4.0)
    want = passes(p, pos, L.HASH_LINEAR, 0)
    for xbits in (0, 2, 4):
        for got, ref in zip(passes(p, pos, L.HASH_MORTON, xbits), want):
            assert np.array_equal(got, ref, equal_nan=True)


# rows of 31..33, 63..65 and more candidates beside ordinary ones, at the seam
# and inside; the Morton order tests every candidate, the linear one takes masks
@pytest.mark.parametrize("cellcount", [1, 2, 3])
@pytest.mark.parametrize("crowd", [0, 31, 32, 33, 64, 150])
@pytest.mark.parametrize("build", [lambda: S.channel_poiseuille(1500, nu=1e-2, seed=3),
                                   lambda: S.channel_peristalsis(1500, 0.3, 1.0, seed=3)],
                         ids=["poiseuille", "peristalsis"])
def test_row_masks_equal_the_tested_rows(device, build, crowd, cellcount):
    sc = build()
    p = sc.params
    p.cellcount = cellcount
    S.finalize(p)
    rng = np.random.default_rng(crowd)
    pos = np.array(sc.pos, np.float32)
    inside = np.flatnonzero(np.abs(pos[:, 1] - np.median(pos[:, 1])) < 0.5 * np.ptp(pos[:, 1]))
    lo = [float(p.world_origin[a]) for a in range(2)]
    pick = rng.permutation(inside)[: 2 * crowd]
    mid = float(np.median(pos[:, 1]))
    for part, x0 in ((pick[:crowd], lo[0] + 0.5 * float(p.world_size[0])), (pick[crowd:], lo[0])):
        pos[part, 0] = x0 + float(p.cell_size[0]) * rng.uniform(0.01, 0.9, len(part))
        pos[part, 1] = mid + float(p.cell_size[1]) * rng.uniform(0.01, 0.9, len(part))
    want = passes(p, pos, L.HASH_MORTON, 0, sc.vel)
    for got, ref in zip(passes(p, pos, L.HASH_LINEAR, 0, sc.vel), want):
        assert np.array_equal(got, ref, equal_nan=True)


# the same for dam breaks whose targets have a lane each (more than 98,304
# rows): clouds of `fill` particles a cell on average, from none to twice that,
# walls among them, so that blocks span one, two and more rows of cells, candidate
# rows fit the density pass's LDS stage or not, and runs hold 64 candidates or
# more and less; at the border of the grid and inside it, with masks and without
@pytest.mark.parametrize("n,fill,cells_x", [(98305, 8, 40), (100003, 22, 12), (98560, 22, 60), (120011, 45, 30),
                                            (98305, 110, 9)])
@pytest.mark.parametrize("border", [False, True])
def test_one_lane_targets_in_irregular_clouds(device, n, fill, cells_x, border):
    sc = S.dambreak3d(dx=0.02)
    p = sc.params
    at = np.zeros(3) if border else np.array([1, 1, 1])
    rng = np.random.default_rng(n + fill)
    rows = -(-n // (fill * cells_x))
    ny = max(int(round(rows ** 0.5)), -(-rows // (int(p.grid_size[2]) - 2)))
    nz = -(-rows // ny)
    span = np.array([cells_x, ny, nz])
    assert (at + span <= [int(g) for g in p.grid_size]).all()
    cells = np.stack(np.meshgrid(*[np.arange(k) for k in span], indexing="ij"), -1).reshape(-1, 3)
    weight = rng.uniform(0.0, 2.0, len(cells))
    pick = cells[rng.choice(len(cells), n, p=weight / weight.sum())]
    pos = np.zeros((n, 4), np.float32)
    cs = np.array([float(c) for c in p.cell_size])
    pos[:, :3] = [float(o) for o in p.world_origin] + cs * (at + pick + rng.uniform(0.01, 0.99, (n, 3)))
    pos[:, 3] = np.where(rng.uniform(size=n) < 0.1, 1.0, 4.0)
    want = passes(p, pos, L.HASH_LINEAR, 0)
    for xbits in (0, 2, 4):
        for got, ref in zip(passes(p, pos, L.HASH_MORTON, xbits), want):
            assert np.array_equal(got, ref, equal_nan=True)
    for order, xbits in ((L.HASH_LINEAR, 0), (L.HASH_MORTON, 4)):
        q = type(p).from_buffer_copy(p)
        q.hash_order, q.morton_xbits = order, xbits
        S.finalize(q)
        s = ParamSystem.from_state(q, pos, None)
        s.set_inrange_masks(False)
        s.update()
        assert np.array_equal(s.getArray(L.ARRAY_ACCELERATION), want[1], equal_nan=True)
        s.close()
