"""The counting sort behind a System's and a batch's step: hash, index and cell
ranges are the stable argsort of the cell keys whatever the particles' order,
cell fill and count, over several steps (the counters are reused)."""
import numpy as np
import pytest

from cmag_amd import _lib as L
from cmag_amd import scenarios as S
from cmag_amd.batch import Batch
from cmag_amd.systems import ParamSystem

pytestmark = pytest.mark.gpu

# edges of a wave and of a workgroup (the offset scan's tiles are cells: below)
COUNTS = [1, 2, 63, 64, 65, 255, 257, 4095, 4097, 30011]


def check_sorted(key, hash_, index, start, end):
    order = np.argsort(key, kind="stable")
    assert np.array_equal(index, order.astype(np.uint32))
    assert np.array_equal(hash_, key[order])
    cells, first, cnt = np.unique(key[order], return_index=True, return_counts=True)
    want = np.full(start.size, L.CELL_EMPTY, np.uint32)
    want[cells] = first
    assert np.array_equal(start, want)
    assert np.array_equal(end[cells], (first + cnt).astype(np.uint32))


def keys_of(p, pos):
    """cell keys in numpy, DIV_CELL rule, linear order (float32 as the hash)"""
    c = [np.floor((pos[:, a] - np.float32(p.world_origin[a])) / np.float32(p.cell_size[a])).astype(np.int64)
         & (int(p.grid_size[a]) - 1) for a in range(3)]
    return ((c[2] * int(p.grid_size[1]) + c[1]) * int(p.grid_size[0]) + c[0]).astype(np.uint32)


def check_system(s, p, steps):
    for _ in range(steps):
        before = s.getArray(L.ARRAY_POSITION)
        s.update()
        arr = [s.getUintArray(a) for a in (L.ARRAY_HASH, L.ARRAY_INDEX, L.ARRAY_CELLSTART, L.ARRAY_CELLEND)]
        check_sorted(keys_of(p, before), *arr)
        assert np.array_equal(s.getArray(L.ARRAY_SORTEDPOS), before[arr[1]])


@pytest.mark.parametrize("n", COUNTS)
@pytest.mark.parametrize("fill", ["lattice", "shuffled", "one_cell", "two_cells"])
def test_system_sort(device, n, fill):
    # the dam break's grid (sub-cell copies too) and the channel's (none)
    for sc, walk in ((S.dambreak3d(dx=0.05), True), (S.channel_poiseuille(3000, nu=1e-2, seed=1), False)):
        p = sc.params
        if fill in ("one_cell", "two_cells") and n > 5000:
            n = 5000  # the neighbour passes test every pair of a cell
        rng = np.random.default_rng(n)
        pos = np.zeros((n, 4), np.float32)
        lo = np.array([float(p.world_origin[a]) for a in range(3)])
        size = np.array([float(p.world_size[a]) for a in range(3)])
        u = rng.uniform(0.1, 0.9, (n, 3))
        if fill == "lattice":
            u = u[np.lexsort((u[:, 0], np.floor(u[:, 1] * 40)))]
        elif fill in ("one_cell", "two_cells"):
            cs = np.array([float(p.cell_size[a]) for a in range(3)]) / size
            at = np.floor(0.4 / cs) * cs
            u = at + cs * (0.2 + 0.6 * rng.uniform(size=(n, 3)))
            if fill == "two_cells":
                u[:, 0] += cs[0] * (rng.uniform(size=n) < 0.5)
        if p.dim == 2:
            u[:, 2] = 0.5
        pos[:, :3] = lo + size * u
        pos[:, 3] = np.where(rng.uniform(size=n) < 0.3, 1.0, 4.0 if walk else 0.0)
        s = ParamSystem.from_state(p, pos, None)
        assert s.subcell_walk == walk
        check_system(s, p, 1)
        # again from the same state: the counters were left clean
        s.setArray(L.ARRAY_POSITION, pos)
        check_system(s, p, 1)
        if walk:  # off and on again: cells that emptied meanwhile hold no counts
            s.set_subcell_walk(False)
            s.setArray(L.ARRAY_POSITION, pos[::-1])
            check_system(s, p, 1)
            s.set_subcell_walk(True)
            half = pos.copy()
            half[: n // 2, 0] += float(p.cell_size[0])
            s.setArray(L.ARRAY_POSITION, half)
            check_system(s, p, 1)
            a = s.getArray(L.ARRAY_ACCELERATION)
            fresh = ParamSystem.from_state(p, half, None)
            zero = np.zeros_like(half)
            s.setArray(L.ARRAY_POSITION, half)
            for arr in (L.ARRAY_VELOCITY, L.ARRAY_VELOCITYLEAPFROG, L.ARRAY_ACCELERATION):
                s.setArray(arr, zero)
            s.update()
            fresh.update()
            a, b = s.getArray(L.ARRAY_ACCELERATION), fresh.getArray(L.ARRAY_ACCELERATION)
            assert np.array_equal(a, b, equal_nan=True)
            fresh.close()
        s.close()


def test_batch_sort(device):
    scen = [S.channel_poiseuille(n, nu=1e-2, seed=n) for n in (1024, 1500, 5003)]
    scen += [S.channel_peristalsis(2000, 0.3, 1.0, seed=3)]
    b = Batch([(sc.params, sc.pos, sc.vel) for sc in scen])
    n, cells = b.num_particles, b.num_cells
    import torch

    class View:
        def __init__(self, ptr, k):
            self.owner = b
            self.__cuda_array_interface__ = {"shape": (k,), "typestr": "<i4", "data": (ptr, False), "version": 2}

    def u32(arr, k):
        return torch.as_tensor(View(b.device_ptr(arr), k), device="cuda").cpu().numpy().view(np.uint32)

    for _ in range(3):
        key, part0, cell0 = [], 0, 0
        for k, sc in enumerate(scen):
            key.append(keys_of(sc.params, b.getArray(k, L.ARRAY_POSITION)) + np.uint32(cell0))
            cell0 += S.num_cells(sc.params)
        b.update()
        b.synchronize()
        check_sorted(np.concatenate(key), u32(L.ARRAY_HASH, n), u32(L.ARRAY_INDEX, n), u32(L.ARRAY_CELLSTART, cells),
                     u32(L.ARRAY_CELLEND, cells))
    b.close()


def on_grid(p, sizes, n, seed, walls):
    """p on a grid of these sizes, and n particles over all of it: half anywhere,
    half in blocks of eight cells, among them the grid's first and last cells"""
    cs = float(p.cell_size[0])
    p.hash_order = L.HASH_LINEAR
    for a, g in enumerate(sizes):
        p.grid_size[a] = g
        p.cell_size[a] = cs
        p.world_origin[a] = 0.0
        p.world_size[a] = g * cs
    S.finalize(p)
    rng = np.random.default_rng(seed)
    g = np.array(sizes)
    cell = rng.integers(0, g, (n, 3))
    near = rng.integers(0, max(n // 64, 1), n // 2)
    corner = rng.integers(0, g, (max(n // 64, 1), 3))
    corner[0], corner[-1] = 0, g - 1
    cell[: n // 2] = np.minimum(corner[near] + rng.integers(0, 2, (n // 2, 3)), g - 1)
    cell[0], cell[-1] = 0, g - 1
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = cs * (cell + rng.uniform(0.2, 0.8, (n, 3)))
    pos[:, 3] = np.where(rng.uniform(size=n) < 0.3, 1.0, 4.0) if walls else 0.0
    return p, pos


# grids of two to eight 16,384-cell tiles whose workgroups sum the counts in
# front of them, of 4,096-cell tiles with totals (from 2^18 cells), and of more
# tiles than a workgroup sums (2^26 cells: the totals are scanned)
@pytest.mark.parametrize("sizes", [(64, 32, 16), (64, 32, 64), (128, 64, 32), (1024, 256, 256)])
@pytest.mark.parametrize("walk", [True, False])
def test_system_sort_on_large_grids(device, sizes, walk):
    n = 5000
    p, pos = on_grid(S.dambreak3d(dx=0.05).params, sizes, n, sizes[2], True)
    s = ParamSystem.from_state(p, pos, None)
    s.set_subcell_walk(walk)
    check_system(s, p, 1)
    dens = np.zeros(n)
    dens[s.getUintArray(L.ARRAY_INDEX)] = s.getArray(L.ARRAY_MEASURES)[:, 0]
    # again from other cells: those that emptied hold no counts
    s.setArray(L.ARRAY_POSITION, pos[::-1].copy())
    check_system(s, p, 1)
    back = np.zeros(n)
    back[s.getUintArray(L.ARRAY_INDEX)] = s.getArray(L.ARRAY_MEASURES)[:, 0]
    # the same neighbours in another order: at most 100 positive terms
    assert np.max(np.abs(back[::-1] - dens) / dens) <= 50 * 6e-8
    s.close()


# cell totals that are no multiple of 16 in each of the offset kernel's forms
@pytest.mark.parametrize("large", [(64, 32, 1), (128, 128, 1), (512, 256, 1)])
def test_batch_sort_ends_in_a_partial_tile(device, large):
    inst = []
    for k, (sizes, n) in enumerate((((2, 4, 1), 30), (large, 3000))):
        p, pos = on_grid(S.channel_poiseuille(1024, nu=1e-2, seed=1).params, sizes, n, k, False)
        inst.append((p, pos, np.zeros_like(pos)))
    b = Batch(inst)
    n, cells = b.num_particles, b.num_cells
    assert cells % 16 == 8
    import torch

    class View:
        def __init__(self, ptr, k):
            self.owner = b
            self.__cuda_array_interface__ = {"shape": (k,), "typestr": "<i4", "data": (ptr, False), "version": 2}

    def u32(arr, k):
        return torch.as_tensor(View(b.device_ptr(arr), k), device="cuda").cpu().numpy().view(np.uint32)

    key, cell0 = [], 0
    for p, pos, _ in inst:
        key.append(keys_of(p, pos) + np.uint32(cell0))
        cell0 += S.num_cells(p)
    b.update()
    b.synchronize()
    check_sorted(np.concatenate(key), u32(L.ARRAY_HASH, n), u32(L.ARRAY_INDEX, n), u32(L.ARRAY_CELLSTART, cells),
                 u32(L.ARRAY_CELLEND, cells))
    b.close()
