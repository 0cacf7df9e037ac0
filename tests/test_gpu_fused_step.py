"""The force pass of channels and small dam breaks integrates its targets; with
stage timing on the two stages run as launches of their own.  The operations are the same, so the states
are the same bit for bit."""
import numpy as np
import pytest

from cmag_amd import _lib as L
from cmag_amd import scenarios as S
from cmag_amd.batch import Batch
from cmag_amd.systems import ParamSystem

pytestmark = pytest.mark.gpu

ARRAYS = (L.ARRAY_POSITION, L.ARRAY_VELOCITY, L.ARRAY_VELOCITYLEAPFROG, L.ARRAY_ACCELERATION)


def scene(kind, n):
    sc = S.channel_poiseuille(n, nu=2e-2, seed=3) if kind == "poiseuille" else S.channel_peristalsis(n, 0.3, 1.2, seed=3)
    vel = np.zeros_like(sc.pos)
    vel[:sc.num_fluid, 0] = 1e-2
    vel[:, 3] = np.arange(len(vel), dtype=np.float32)  # w is carried along
    return sc.params, sc.pos, vel


def states(s, arrays=ARRAYS):
    return [np.asarray(s.getArray(a)) for a in arrays]


@pytest.mark.parametrize("kind", ["poiseuille", "peristalsis"])
@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("n", [1000, 2500])
def test_system(device, kind, moving, n):
    p, pos, vel = scene(kind, n)
    if moving:
        p = p.copy()
        p.is_boundary_configuration = 0
        p.wall_velocity = 1
    out = []
    for timing in (False, True):
        s = ParamSystem(p, pos.shape[0])
        for a, x in zip(ARRAYS, (pos, vel, vel)):
            s.setArray(a, x)
        s.enable_timing(timing)
        for _ in range(3):
            s.update()
        out.append(states(s))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("cells", [3, 12])
@pytest.mark.parametrize("order,xbits", [(L.HASH_LINEAR, 0), (L.HASH_MORTON, 3)])
def test_small_dam_break(device, cells, order, xbits):
    sc = S.dambreak3d(dx=0.4 / cells, hash_order=order, morton_xbits=xbits)
    rng = np.random.default_rng(cells)
    vel = rng.normal(scale=0.3, size=sc.pos.shape).astype(np.float32)  # w of every particle is carried along
    out = []
    for timing in (False, True):
        s = ParamSystem(sc.params, sc.pos.shape[0])
        for a, x in zip(ARRAYS, (sc.pos, vel, vel[::-1].copy())):
            s.setArray(a, x)
        s.enable_timing(timing)
        for _ in range(3):
            s.update()
        out.append(states(s))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("kind", ["poiseuille", "peristalsis", "dambreak"])
def test_runs_of_several_steps_replay_the_single_steps(device, kind):
    """run() launches several captured steps at a time once counts repeat (up to
    16): every state along growing, shrinking and mixed counts, with eager steps,
    array writes and parameter changes between them, equals the eager steps' """
    if kind == "dambreak":
        sc = S.dambreak3d(dx=0.4 / 7)
        p, pos, vel = sc.params, sc.pos, np.zeros_like(sc.pos)
    else:
        p, pos, vel = scene(kind, 1000)
    a, b = (ParamSystem(p, pos.shape[0]) for _ in range(2))
    for s in (a, b):
        for arr, x in zip(ARRAYS, (pos, vel, vel)):
            s.setArray(arr, x)
    for k, steps in enumerate([3, 3, 3, 10, 10, 3, 3, 0, 40, 40, 1, 1, 17, 17, 2, 10]):
        a.run(steps)
        b.run(steps, use_graph=False)
        if k % 5 == 2:
            a.update()
            b.update()
        if k == 6:
            for s in (a, b):
                s.setArray(L.ARRAY_VELOCITY, vel)
        if k == 8:
            q = a.params.copy()
            q.gravity[0] = 1e-3
            a.set_params(q)
            b.set_params(q)
        for x, y in zip(states(a), states(b)):
            assert np.array_equal(x, y, equal_nan=True), (k, steps)
        assert a.getElapsedTime() == b.getElapsedTime()


def test_batch(device):
    inst = [scene(k, n) for k, n in (("poiseuille", 1000), ("peristalsis", 1100), ("poiseuille", 1500))]
    out = []
    for timing in (False, True):
        b = Batch(inst)
        b.enable_timing(timing)
        for _ in range(3):
            b.update()
        out.append([np.asarray(b.getArray(k, a)) for k in range(3) for a in ARRAYS])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
