"""The workloads this framework is timed on, through its public entry points.

Each case stands for work that a user's program has it do:

  channel     one 2-D Poiseuille channel (ParamSystem), stepped by update() or
              by run() with its captured step
  peristalsis one 2-D channel with moving sinusoidal walls, likewise
  dam2d       the reference's own 2-D dam break (DamBreakSystem on its default
              cells), stepped by update() as its demo does
  dam3d       the 3-D dam break behind its gate (Tait, wall particles), linear
              or Z-order cells
  batch       many uneven channels, half Poiseuille, half peristaltic, in one
              launch sequence per step (Batch)
  adjoint     forward and backward of a channel rollout: the gradient of a
              velocity-profile loss in viscosity and body force
  launchers   the stage launchers of the C ABI over a caller's own buffers:
              hash, sort, reorder, density, force

Initial states are lattices with seeded jitter and a smooth velocity field with
seeded noise (a flow under way rather than a start from rest).  exact() restates
the step in 64 bits with plain torch: pair lists from the cells, then the sums.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from cmag_amd import _lib as L
from cmag_amd import scenarios as S
from cmag_amd.adjoint import ChannelRollout, profile_loss
from cmag_amd.batch import Batch
from cmag_amd.systems import DamBreakSystem, ParamSystem

DEV = "cuda"
STATE = (L.ARRAY_POSITION, L.ARRAY_VELOCITY, L.ARRAY_VELOCITYLEAPFROG)


# ---------------------------------------------------------------- the cases
def listed() -> list[dict]:
    return [
        # the plain 2-D channel of the steady-profile check: 2,048 fluid particles, a long run of captured steps
        {"name": "channel_2k", "kind": "channel", "n": 2240, "nu": 1e-2, "steps": 10, "graph": True},
        # the same physics at the size of a parameter study, stepped one update() at a time between a program's own work
        {"name": "channel_17k", "kind": "channel", "n": 17500, "nu": 2e-2, "steps": 1, "graph": False},
        # a finely resolved single channel, an odd count
        {"name": "channel_200k", "kind": "channel", "n": 200003, "nu": 5e-3, "steps": 2, "graph": True},
        # one peristaltic channel, captured steps
        {"name": "peristalsis_9k", "kind": "peristalsis", "n": 9001, "amp": 0.3, "wl": 1.2, "steps": 10, "graph": True},
        # the reference demo's dam break: 128 x 128 fluid particles on cells of one particle spacing
        {"name": "dam2d_17k", "kind": "dam2d", "nx": 128, "ny": 128},
        # a coarse 3-D dam break, captured steps
        {"name": "dam3d_16k", "kind": "dam3d", "cells": 20, "order": "morton", "xbits": 4, "alpha": 0.38, "steps": 2,
         "graph": True},
        # the 1M-particle 3-D dam break on linear cells
        {"name": "dam3d_1m", "kind": "dam3d", "cells": 80, "order": "linear", "xbits": 0, "alpha": 0.01, "steps": 1,
         "graph": False},
        # the 16M-particle 3-D dam break on Z-order cells: the largest workload
        {"name": "dam3d_16m", "kind": "dam3d", "cells": 202, "order": "morton", "xbits": 7, "alpha": 0.01, "steps": 1,
         "graph": False},
        # a handful of small channels, one eager batched step
        {"name": "batch_24", "kind": "batch", "m": 24, "mix": 7, "n_lo": 1024, "n_hi": 8192, "steps": 1, "graph": False},
        # 256 channels of 1k to 64k particles, one graph of ten steps
        {"name": "batch_256", "kind": "batch", "m": 256, "mix": 20240, "n_lo": 1024, "n_hi": 65536, "steps": 10,
         "graph": True},
        # the differentiable run: 16k particles, 200 steps, checkpoints every 20
        {"name": "adjoint_17k", "kind": "adjoint", "nx": 128, "ny": 128, "steps": 200, "every": 20},
        # the stage launchers over a caller's buffers, 3-D dam break, linear cells
        {"name": "launchers_300k", "kind": "launchers", "cells": 45, "order": "linear", "xbits": 0},
    ]


def _log(rng, lo, hi) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(["channel", "channel", "peristalsis", "dam2d", "dam3d", "dam3d", "dam3d", "batch", "adjoint",
                       "launchers"])
    steps, graph = rng.choice([(1, False), (1, True), (2, False), (4, True), (10, True)])
    order = rng.choice(["linear", "morton"])
    xbits = rng.choice([0, 2, 4, 7]) if order == "morton" else 0
    if kind == "channel":
        return {"kind": kind, "n": int(_log(rng, 1000, 250000)), "nu": _log(rng, 1e-3, 1e-1), "steps": steps,
                "graph": graph}
    if kind == "peristalsis":
        return {"kind": kind, "n": int(_log(rng, 1000, 65536)), "amp": rng.uniform(0.1, 0.5),
                "wl": rng.uniform(0.5, 2.0), "steps": steps, "graph": graph}
    if kind == "dam2d":
        return {"kind": kind, "nx": int(_log(rng, 16, 256)), "ny": int(_log(rng, 16, 256))}
    if kind == "dam3d":
        cells = int(_log(rng, 8, 160))
        return {"kind": kind, "cells": cells, "order": order, "xbits": xbits, "alpha": 0.38 if cells < 50 else 0.01,
                "steps": min(steps, 2) if cells < 50 else 1, "graph": graph}
    if kind == "batch":
        n_hi = int(_log(rng, 4096, 65536))
        return {"kind": kind, "m": int(_log(rng, 2, 200)), "mix": rng.randrange(1 << 20), "n_lo": 1024, "n_hi": n_hi,
                "steps": steps, "graph": graph}
    if kind == "adjoint":
        return {"kind": kind, "nx": rng.choice([16, 32, 64, 128]), "ny": 2 * rng.randrange(16, 75),
                "steps": rng.randrange(10, 200), "every": rng.randrange(3, 24)}
    return {"kind": kind, "cells": int(_log(rng, 8, 70)), "order": order, "xbits": xbits}


# ---------------------------------------------------------------- scenarios (host, without the seed)
def _key(case: dict) -> tuple:
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "steps", "graph", "every")))


def _order(case: dict) -> dict:
    return dict(hash_order=L.HASH_MORTON if case["order"] == "morton" else L.HASH_LINEAR, morton_xbits=case["xbits"])


@functools.lru_cache(maxsize=16)
def _scenarios(key: tuple) -> list:
    c = dict(key)
    if c["kind"] == "channel":
        return [S.channel_poiseuille(c["n"], c["nu"], seed=1, jitter=0.0)]
    if c["kind"] == "peristalsis":
        return [S.channel_peristalsis(c["n"], c["amp"], c["wl"], seed=1, jitter=0.0)]
    if c["kind"] in ("dam3d", "launchers"):
        return [S.dambreak3d(dx=0.4 / c["cells"], alpha=c.get("alpha", 0.38), jitter=0.0, **_order(c))]
    if c["kind"] == "batch":
        return S.channel_batch(m=c["m"], seed=c["mix"], n_lo=c["n_lo"], n_hi=c["n_hi"])
    if c["kind"] == "adjoint":
        return [S.poiseuille_channel(nx=c["nx"], ny=c["ny"], nu=2e-2, jitter=0.0)]
    raise ValueError(c["kind"])


def _scen(case: dict) -> list:
    return _scenarios(_key(case))


@functools.lru_cache(maxsize=4)
def _lattice(key: tuple) -> torch.Tensor:
    return torch.as_tensor(_scenarios(key)[0].pos, device=DEV)


def _dam2d(case: dict) -> tuple:
    nx, ny = case["nx"], case["ny"]
    r = 1.0 / 256  # the reference's particle mass belongs to this radius
    gx = 1 << max(6, (4 * nx - 1).bit_length())
    gy = 1 << max(5, (2 * ny - 1).bit_length())
    return (nx, ny, 1), 1, (gx, gy, 4), r


def _count(case: dict) -> int:
    if case["kind"] == "dam2d":
        f, bo, g, _ = _dam2d(case)
        return f[0] * f[1] + g[0] * bo + 2 * (g[1] - bo) * bo
    return sum(int(sc.pos.shape[0]) for sc in _scen(case))


# ---------------------------------------------------------------- initial states (on the GPU, from the seed)
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _noise(g: torch.Generator, n: int) -> torch.Tensor:
    return torch.rand((n, 3), generator=g, device=DEV, dtype=torch.float32) * 2 - 1


def _channel_state(sc, pos: torch.Tensor, g: torch.Generator):
    """jittered lattice, x-velocity over the channel's height with 1 % noise"""
    peri = sc.params.system == L.SYS_PERISTALSIS
    fl = (pos[:, 3:4] == 0.0).float()
    nz = _noise(g, pos.shape[0])
    nz[:, 2] = 0.0
    pos = pos.clone()
    pos[:, :3] += fl * nz * (1e-3 * sc.meta["dx"])
    s = torch.clamp(2.0 * pos[:, 1] / sc.meta["width"], -1.0, 1.0)
    u = (float(sc.params.wave_speed) if peri else sc.meta["vmax"]) * (1.0 - s * s)
    vel = torch.zeros_like(pos)
    nv = _noise(g, pos.shape[0])
    vel[:, 0] = fl[:, 0] * u * (1.0 + 0.01 * nv[:, 0])
    vel[:, 1] = fl[:, 0] * u * 0.01 * nv[:, 1]
    return pos, vel


def _dam_state(pos: torch.Tensor, g: torch.Generator, dx: float, lo, size, speed: float, planar: bool):
    """a column under way: 1 % jitter, one roll of the given speed, 2 % noise"""
    fl = (pos[:, 3:4] == 4.0).float()
    nz, nv = _noise(g, pos.shape[0]), _noise(g, pos.shape[0])
    if planar:
        nz[:, 2] = nv[:, 2] = 0.0
    pos = pos.clone()
    pos[:, :3] += fl * nz * (0.01 * dx)
    x, y = math.pi * (pos[:, 0] - lo[0]) / size[0], math.pi * (pos[:, 1] - lo[1]) / size[1]
    vel = torch.zeros_like(pos)
    vel[:, 0] = speed * torch.sin(x) * torch.cos(y)
    vel[:, 1] = -speed * (size[1] / size[0]) * torch.cos(x) * torch.sin(y)
    vel[:, :3] = fl * (vel[:, :3] + 0.02 * speed * nv)
    return pos, vel


def _state(case: dict, seed: int) -> tuple:
    """(params, pos, vel) of a single system, on the GPU"""
    g = _gen(seed)
    sc = _scen(case)[0]
    pos = _lattice(_key(case))
    if case["kind"] in ("dam3d", "launchers"):
        return (sc.params,) + _dam_state(pos, g, sc.meta["dx"], (0.0, 0.0), sc.meta["column"], 0.5, False)
    return (sc.params,) + _channel_state(sc, pos, g)


def _batch_state(case: dict, seed: int) -> list:
    scen = _scen(case)
    g = _gen(seed)
    out = []
    for sc in scen:
        pos, vel = _channel_state(sc, torch.as_tensor(sc.pos, device=DEV), g)
        out.append((sc.params, pos, vel))
    return out


class _View:
    """device memory that a getter of the framework lends, as a tensor's source; the memory is the owner's and goes
    with it, so the view (and with it every tensor over it) keeps the owner"""

    def __init__(self, owner, ptr: int, n: int):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n, 4), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _borrowed(owner, n: int) -> list:
    return [torch.as_tensor(_View(owner, owner.device_ptr(a), n), device=DEV) for a in STATE]


def _fill(system, pos: torch.Tensor, vel: torch.Tensor) -> None:
    torch.cuda.synchronize()
    for a, t in zip(STATE, (pos, vel, vel)):
        system.copy_from_device(a, t.data_ptr())
    system.synchronize()


# ---------------------------------------------------------------- prepare, run
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    st = {"case": case}
    if kind == "dam2d":
        fluid, bo, grid, r = _dam2d(case)
        s = DamBreakSystem(fluid, bo, grid, r, False)
        s.reset()
        p = s.params
        pos = torch.as_tensor(s.getArray(DamBreakSystem.POSITION), device=DEV)
        lo = [float(p.clamp_lo[0]), float(p.clamp_lo[1])]
        pos, vel = _dam_state(pos, _gen(seed), 2 * r, lo, (fluid[0] * 2 * r, fluid[1] * 2 * r), 0.5, True)
        _fill(s, pos, vel)
        st.update(system=s, out=_borrowed(s, int(pos.shape[0])))
    elif kind in ("channel", "peristalsis", "dam3d"):
        p, pos, vel = _state(case, seed)
        s = ParamSystem(p, int(pos.shape[0]))
        _fill(s, pos, vel)
        st.update(system=s, out=_borrowed(s, int(pos.shape[0])))
    elif kind == "batch":
        b = Batch([(p, pos.cpu().numpy(), vel.cpu().numpy()) for p, pos, vel in _batch_state(case, seed)])
        st.update(system=b, out=_borrowed(b, b.num_particles))
    elif kind == "adjoint":
        p, pos, vel, mu, grav, target = _adjoint_inputs(case, seed)
        r = ChannelRollout(p, pos.cpu().numpy(), vel.cpu().numpy(), steps=case["steps"],
                           checkpoint_every=case["every"])
        st.update(rollout=r, mu=mu, grav=grav, target=target)
    else:
        p, pos, vel = _state(case, seed)
        n, cells = int(pos.shape[0]), S.num_cells(p)
        nbytes = int(L.lib().cmag_sort_scratch_bytes(n, S.key_bits(p)))
        u = lambda k: torch.zeros(k, dtype=torch.int32, device=DEV)  # noqa: E731
        f = lambda: torch.zeros((n, 4), dtype=torch.float32, device=DEV)  # noqa: E731
        st.update(params=p, n=n, cells=cells, bits=S.key_bits(p), pos=pos, vel=vel, hash=u(n), index=u(n),
                  start=u(cells), end=u(cells), spos=f(), svel=f(), meas=f(), acc=f(), nbytes=nbytes,
                  scratch=torch.empty(nbytes, dtype=torch.uint8, device=DEV))
    return st


def _launchers(st: dict) -> dict:
    p, n = C.byref(st["params"]), st["n"]
    d = {k: v.data_ptr() for k, v in st.items() if isinstance(v, torch.Tensor)}
    L.call("cmag_calc_hash", p, d["pos"], d["hash"], d["index"], n, None)
    L.call("cmag_sort_by_key", d["hash"], d["index"], n, st["bits"], d["scratch"], st["nbytes"], None)
    L.call("cmag_reorder_find_cell_start", d["start"], d["end"], d["spos"], d["svel"], d["hash"], d["index"], d["pos"],
           d["vel"], n, st["cells"], None)
    L.call("cmag_density", p, d["meas"], d["spos"], d["start"], d["end"], n, None)
    L.call("cmag_force", p, d["acc"], d["meas"], d["spos"], d["svel"], d["index"], d["start"], d["end"], n, None)
    return {k: st[k] for k in ("hash", "index", "start", "spos", "svel", "meas", "acc")}


def run(st: dict):
    case = st["case"]
    kind = case["kind"]
    if kind == "adjoint":
        mu = st["mu"].clone().requires_grad_(True)
        grav = st["grav"].clone().requires_grad_(True)
        r = st["rollout"]
        pos, vel = r(mu, grav)
        profile_loss(pos, vel, r.params, st["target"], len(st["target"])).backward()
        return {"pos": pos.detach(), "vel": vel.detach(), "mu": mu.grad, "grav": grav.grad}
    if kind == "launchers":
        return _launchers(st)
    s = st["system"]
    if kind == "dam2d":
        s.update()
    elif case["graph"]:
        s.run(case["steps"])
    else:
        for _ in range(case["steps"]):
            s.update()
    return dict(zip(("pos", "vel", "velLF"), st["out"]))


def work(case: dict) -> dict:
    n = _count(case)
    kind = case["kind"]
    # per particle and step: position, velocity and leapfrog velocity read and written; in-range neighbours at the
    # lattice spacing, about 12 operations for a density term and 40 for a force term
    nb = 73.6 if kind in ("dam3d", "launchers") else 28.3 if kind in ("peristalsis", "dam2d") else 21.2
    steps = case.get("steps", 1)
    if kind == "launchers":
        return {"bytes": (32 + 8 + 32 + 16 + 16) * n + 4 * S.num_cells(_scen(case)[0].params), "flops": 52 * nb * n}
    if kind == "adjoint":
        return {"bytes": 3 * 96 * n * steps, "flops": (2 * 52 + 100) * nb * n * steps}
    return {"bytes": 96 * n * steps, "flops": 52 * nb * n * steps}


def _adjoint_inputs(case: dict, seed: int):
    p, pos, vel = _state(case, seed)
    p = p.copy()
    g = _gen(seed + 1)
    u = torch.rand(2, generator=g, device=DEV, dtype=torch.float64).cpu()
    nu, vmax = 1e-2, 1e-2
    p.mu = 1000.0 * nu
    mu = torch.tensor(1000.0 * nu * (0.9 + 0.2 * float(u[0])), dtype=torch.float32)
    grav = torch.tensor([8.0 * nu * vmax * (0.8 + 0.4 * float(u[1])), 0.0, 0.0], dtype=torch.float32)
    bins = case["ny"] // 2  # two lattice rows a bin, so that no particle starts near a bin's edge
    y = (np.arange(bins) + 0.5) / bins
    target = 0.8 * vmax * 4.0 * y * (1.0 - y)
    return p, pos, vel, mu, grav, target


# ---------------------------------------------------------------- the same in 64 bits
class _Par:
    """the parameter blocks of one or several systems as 64-bit tensors, one value a system, spread over its particles"""

    NAMES = ("particle_radius", "smoothing_radius", "particle_mass", "rest_density", "soundspeed", "B", "gamma",
             "delta_time", "boundary_damping", "mu", "alpha", "kernel_coeff", "grad_coeff", "right_boundary", "lj_D",
             "lj_a", "wall_top", "wall_bottom", "beta_max", "amplitude", "wave_speed", "wave_k")
    AXES = ("world_origin", "cell_size", "world_size", "gravity", "clamp_lo", "clamp_hi")

    def __init__(self, blocks, counts):
        self.inst = torch.repeat_interleave(torch.arange(len(blocks), device=DEV), torch.tensor(counts, device=DEV))
        spread = (lambda v: torch.tensor(v, dtype=torch.float64, device=DEV)[self.inst]) if len(blocks) > 1 else (
            lambda v: torch.tensor(v[0], dtype=torch.float64, device=DEV))
        for k in self.NAMES:
            setattr(self, k, spread([float(getattr(b, k)) for b in blocks]))
        for k in self.AXES:
            setattr(self, k, [spread([float(getattr(b, k)[a]) for b in blocks]) for a in range(3)])
        self.many = len(blocks) > 1
        self.blocks = blocks
        self.system = [int(b.system) for b in blocks]
        self.peri_inst = spread([1.0 if b.system == L.SYS_PERISTALSIS else 0.0 for b in blocks]) > 0
        self.is_dam = self.system[0] == L.SYS_DAMBREAK
        self.dim = int(blocks[0].dim)
        self.cc = max(int(b.cellcount) for b in blocks)
        self.periodic = [int(blocks[0].periodic_mask) >> a & 1 for a in range(3)]
        self.grid = [[int(b.grid_size[a]) for b in blocks] for a in range(3)]
        self.half = int(blocks[0].gridpos_rule) != L.GRIDPOS_DIV_CELL
        sizes = [self.grid[0][k] * self.grid[1][k] * self.grid[2][k] for k in range(len(blocks))]
        self.cells = sum(sizes)
        ti = lambda v: torch.tensor(v, device=DEV, dtype=torch.int64)[self.inst]  # noqa: E731
        self.fluid_y = spread([float(b.fluid_size[1]) for b in blocks])
        self.g = [ti(self.grid[a]) for a in range(3)]
        self.cell0 = ti([sum(sizes[:k]) for k in range(len(blocks))])

    def at(self, v, i):
        return v[i] if self.many else v


def _cell_of(P: _Par, pos: torch.Tensor):
    """cell coordinates by the hash's own rule, in the 32 bits it is defined in"""
    x = pos[:, :3].float()
    out = []
    for a in range(3):
        d = x[:, a] - P.world_origin[a].float()
        one = torch.ones(1, device=DEV, dtype=torch.float32)
        out.append(torch.floor(d * 0.5 / (P.particle_radius.float() * one) if P.half else
                               d / (P.cell_size[a].float() * one)).long())
    return out


def _pairs(P: _Par, pos: torch.Tensor, keep, chunk: int = 1 << 20):
    """yields (i, j, image shift along x) for the stencil pairs that keep(i, j, r2, r2max) takes"""
    n = pos.shape[0]
    c = _cell_of(P, pos)
    key = lambda x, y, z, i: P.cell0[i] + ((z & (P.g[2][i] - 1)) * P.g[1][i] + (y & (P.g[1][i] - 1))) * P.g[0][i] + (  # noqa: E731
        x & (P.g[0][i] - 1))
    every = torch.arange(n, device=DEV)
    k = key(c[0], c[1], c[2], every)
    k, order = torch.sort(k, stable=True)
    first = torch.searchsorted(k, torch.arange(P.cells + 1, device=DEV))
    x64 = pos[:, :3].double()
    zs = range(-P.cc, P.cc + 1) if P.dim == 3 else (0,)
    for lo in range(0, n, chunk):
        got = []
        i0 = every[lo:lo + chunk]
        for dz in zs:
            for dy in range(-P.cc, P.cc + 1):
                for dx in range(-P.cc, P.cc + 1):
                    cx, cy, cz = c[0][i0] + dx, c[1][i0] + dy, c[2][i0] + dz
                    if P.periodic[0]:
                        shift = (cx > P.g[0][i0] - 1).long() - (cx < 0).long()
                    else:
                        shift = torch.zeros_like(cx)
                    cell = key(cx, cy, cz, i0)
                    s, e = first[cell], first[cell + 1]
                    for t in range(int((e - s).max())):
                        ok = torch.nonzero(s + t < e).squeeze(1)
                        i, j, sh = i0[ok], order[s[ok] + t], shift[ok]
                        d = x64[i] - x64[j]
                        d[:, 0] -= sh * P.at(P.world_size[0], i)
                        r2 = (d * d).sum(1)
                        h = P.at(P.smoothing_radius, i)
                        m = torch.nonzero(keep(i, j, r2, 4 * h * h)).squeeze(1)
                        got.append((i[m], j[m], sh[m]))
        yield tuple(torch.cat([q[a] for q in got]) for a in range(3))


def _near(i, j, r2, r2max):
    return (i != j) & (r2 < r2max)


def _pressure(P: _Par, rho: torch.Tensor) -> torch.Tensor:
    eos = int(P.blocks[0].eos)
    tait = P.B * ((rho / P.rest_density) ** P.gamma - 1)
    if P.many:
        return torch.where(P.peri_inst, 50 * P.soundspeed * rho, tait)
    return tait if eos == L.EOS_TAIT else 50 * P.soundspeed * rho if eos == L.EOS_LINEAR_50C else P.soundspeed ** 2 * rho


def _diff(P: _Par, x, i, j, sh):
    d = x[i] - x[j]
    return torch.stack([d[:, 0] - sh * P.at(P.world_size[0], i), d[:, 1], d[:, 2]], 1)


def _density(P: _Par, x, w, lists):
    rho = P.kernel_coeff * P.particle_mass * torch.ones(x.shape[0], dtype=torch.float64, device=DEV)
    for i, j, sh in lists:
        r = _diff(P, x, i, j, sh)
        q = torch.sqrt((r * r).sum(1)) / P.at(P.smoothing_radius, i)
        t = 1 - q / 2
        rho = rho.index_add(0, i, P.at(P.kernel_coeff * P.particle_mass, i) * t ** 4 * (2 * q + 1))
    if not P.is_dam:  # Poiseuille walls hold the rest density
        rho = torch.where((w == 1) & ~P.peri_inst, P.rest_density, rho)
    return rho


def _gradient(P: _Par, r, i):
    d = torch.sqrt((r * r).sum(1))
    q = d / P.at(P.smoothing_radius, i)
    t = 1 - q / 2
    return P.at(P.grad_coeff, i) * (t ** 4 - t ** 3 * (2 * q + 1)) / d


def _channel_acc(P: _Par, x, lf, w, lists, mu=None):
    rho = _density(P, x, w, lists)
    pt = _pressure(P, rho) / rho ** 2
    acc = torch.zeros_like(x)
    mu = P.mu if mu is None else mu
    for i, j, sh in lists:
        r = _diff(P, x, i, j, sh)
        g = _gradient(P, r, i)
        m = P.at(P.particle_mass, i)
        V = lf[i] - lf[j]
        wall = (w[j] == 1) & ~P.at(P.peri_inst, i)
        top, bot = P.at(P.wall_top, i), P.at(P.wall_bottom, i)
        yi, yj = x[i, 1], x[j, 1]
        up, dn = wall & (yj > top), wall & (yj < bot)
        one = torch.ones_like(yi)
        bu = torch.minimum(P.at(P.beta_max, i), 1 + (yj - top) / torch.where(up, top - yi, one))
        bd = torch.minimum(P.at(P.beta_max, i), 1 + (bot - yj) / torch.where(dn, yi - bot, one))
        V = torch.where(up[:, None], bu[:, None] * lf[i], torch.where(dn[:, None], bd[:, None] * lf[i], V))
        f = (-m * (pt[i] + pt[j]) * g)[:, None] * r + (2 * m * (P.at(mu, i) if mu is P.mu else mu) * g / (rho[i] * rho[j]))[:, None] * V
        acc = acc.index_add(0, i, f)
    return acc


def _integrate_free(P: _Par, x, v, acc, grav):
    dt = P.delta_time[:, None] if P.many else P.delta_time
    nv = v + (acc + grav) * dt
    return x + nv * dt, nv, (v + nv) / 2


def _channel_exact(blocks, counts, pos, vel, steps):
    P = _Par(blocks, counts)
    w = pos[:, 3].double()
    x, v, lf = pos[:, :3].double(), vel[:, :3].double(), vel[:, :3].double()
    grav = torch.stack([g.expand(x.shape[0]) for g in P.gravity], 1)
    fluid = (w == 0)[:, None]
    t = torch.zeros_like(P.delta_time)
    for _ in range(steps):
        lists = list(_pairs(P, x, _near))
        acc = _channel_acc(P, x, lf, w, lists)
        nx, nv, nl = _integrate_free(P, x, v, acc, grav)
        lo, size = P.world_origin[0], P.world_size[0]
        px = torch.where(nx[:, 0] > lo + size, nx[:, 0] - size, nx[:, 0])
        px = torch.where(P.peri_inst & (px < lo), px + size, px)
        nx = torch.cat([px[:, None], nx[:, 1:]], 1)
        # peristaltic walls ride the sinusoid
        arg = P.wave_k * ((x[:, 0] - lo) - P.wave_speed * t)
        ny, r = P.fluid_y, P.particle_radius
        s, dv = P.amplitude * torch.sin(arg), P.amplitude * torch.cos(arg) * P.wave_k * -P.wave_speed
        wy = torch.where(w > 0, -ny * r + s - r * (w - 1), ny * r - s + r * (-w - 1))
        wv = torch.where(w > 0, dv, -dv)
        move = P.peri_inst & (w != 0)
        wx = torch.where(move[:, None], torch.stack([x[:, 0], wy, x[:, 2]], 1), x)
        zero = torch.zeros_like(wv)
        wvel = torch.where(move[:, None], torch.stack([zero, wv, zero], 1), v)
        wlf = torch.where(move[:, None], torch.stack([zero, wv, zero], 1), lf)
        x, v, lf = torch.where(fluid, nx, wx), torch.where(fluid, nv, wvel), torch.where(fluid, nl, wlf)
        t = t + P.delta_time
    return _rows(pos, vel, x, v, lf)


def _rows(pos, vel, x, v, lf):
    w, vw = pos[:, 3:4].double(), vel[:, 3:4].double()
    return {"pos": torch.cat([x, w], 1), "vel": torch.cat([v, vw], 1), "velLF": torch.cat([lf, vw], 1)}


def _dam_acc(P: _Par, x, lf, w):
    wall = w != 4
    lists = []

    def keep(i, j, r2, r2max):
        return (i != j) & ((r2 < r2max) | (wall[j] & ~wall[i]))

    rho = P.kernel_coeff * P.particle_mass * torch.ones(x.shape[0], dtype=torch.float64, device=DEV)
    for i, j, sh in _pairs(P, x, keep):
        lists.append((i, j))
        r = x[i] - x[j]
        q = torch.sqrt((r * r).sum(1)) / P.smoothing_radius
        t = torch.clamp(1 - q / 2, min=0)
        rho.index_add_(0, i, P.kernel_coeff * P.particle_mass * t ** 4 * (2 * q + 1))
    p = _pressure(P, rho)
    pt = p / rho ** 2
    h = P.smoothing_radius
    acc = torch.zeros_like(x)
    for i, j in lists:
        m = torch.nonzero(~wall[i]).squeeze(1)
        i, j = i[m], j[m]
        r = x[i] - x[j]
        r2 = (r * r).sum(1)
        lj = P.lj_a ** 2 / r2
        f = P.lj_D * (lj ** 6 - lj ** 3) / r2
        vr = ((lf[i] - lf[j]) * r).sum(1)
        av = -2 * P.alpha * h * P.soundspeed * torch.clamp(vr, max=0) / ((rho[i] + rho[j]) * (r2 + 0.001 * h * h))
        g = -P.particle_mass * (pt[i] + pt[j] + av) * _gradient(P, r, i)
        f = torch.where(wall[j], f, torch.where(r2 < 4 * h * h, g, torch.zeros_like(g)))
        acc.index_add_(0, i, f[:, None] * r)
    return rho, p, acc


def _dam_exact(block, pos, vel, steps):
    P = _Par([block], [pos.shape[0]])
    w = pos[:, 3].double()
    x, v, lf = pos[:, :3].double(), vel[:, :3].double(), vel[:, :3].double()
    grav = torch.stack([g.expand(x.shape[0]) for g in P.gravity], 1)
    fluid = (w == 4)[:, None]
    for _ in range(steps):
        nx, nv, nl = _integrate_free(P, x, v, _dam_acc(P, x, lf, w)[2], grav)
        lo = torch.stack(P.clamp_lo)
        hi = torch.stack([P.right_boundary, P.clamp_hi[1], P.clamp_hi[2]])
        out = (nx < lo) | (nx > hi)
        nv = torch.where(out, nv * P.boundary_damping, nv)
        nx = torch.minimum(torch.maximum(nx, lo), hi)
        x, v, lf = torch.where(fluid, nx, x), torch.where(fluid, nv, v), torch.where(fluid, nl, lf)
    return _rows(pos, vel, x, v, lf)


def _launchers_exact(case, seed):
    block, pos, vel = _state(case, seed)
    P = _Par([block], [pos.shape[0]])
    w = pos[:, 3].double()
    rho, p, acc = _dam_acc(P, pos[:, :3].double(), vel[:, :3].double(), w)
    zero = torch.zeros_like(rho)
    c = _cell_of(P, pos)
    g = P.grid
    if case["order"] == "linear":
        order = torch.argsort(((c[2] & (g[2][0] - 1)) * g[1][0] + (c[1] & (g[1][0] - 1))) * g[0][0] + (
            c[0] & (g[0][0] - 1)), stable=True)
        meas = torch.stack([rho, p, zero, zero], 1)[order]
    else:
        meas = None
    return {"hash": None, "index": None, "start": None, "spos": None, "svel": None, "meas": meas,
            "acc": torch.cat([acc, zero[:, None]], 1)}


def _adjoint_exact(case, seed):
    p, pos, vel, mu, grav, target = _adjoint_inputs(case, seed)
    P = _Par([p], [pos.shape[0]])
    w = pos[:, 3].double()
    fluid = (w == 0)[:, None]
    lo, size = P.world_origin[0], P.world_size[0]
    mu = mu.double().to(DEV).requires_grad_(True)
    grav = grav.double().to(DEV).requires_grad_(True)

    def step(x, v, lf, lists):
        nx, nv, nl = _integrate_free(P, x, v, _channel_acc(P, x, lf, w, lists, mu), grav)
        wrap = torch.where(nx[:, 0] > lo + size, size, torch.zeros_like(nx[:, 0]))
        nx = torch.cat([(nx[:, 0] - wrap)[:, None], nx[:, 1:]], 1)
        return torch.where(fluid, nx, x), torch.where(fluid, nv, v), torch.where(fluid, nl, lf)

    states = [(pos[:, :3].double(), vel[:, :3].double(), vel[:, :3].double())]
    pairs = []
    with torch.no_grad():
        for _ in range(case["steps"]):
            pairs.append(list(_pairs(P, states[-1][0], _near)))
            states.append(step(*states[-1], pairs[-1]))
    x, v, _ = states[-1]
    v = v.clone().requires_grad_(True)
    fl, nb = w == 0, len(target)
    b = torch.clamp(torch.floor((x[fl, 1] - P.wall_bottom) / ((P.wall_top - P.wall_bottom) / nb)).long(), 0, nb - 1)
    cnt = torch.zeros(nb, dtype=torch.float64, device=DEV).index_add(0, b, torch.ones_like(x[fl, 0]))
    prof = torch.zeros(nb, dtype=torch.float64, device=DEV).index_add(0, b, v[fl, 0]) / torch.clamp(cnt, min=1)
    loss = (((prof - torch.as_tensor(target, device=DEV)) ** 2) * (cnt > 0)).sum()
    bar = [torch.zeros_like(x), torch.autograd.grad(loss, v)[0], torch.zeros_like(x)]
    dmu, dg = torch.zeros_like(mu), torch.zeros_like(grav)
    for t in reversed(range(case["steps"])):
        ins = [s.detach().requires_grad_(True) for s in states[t]]
        out = step(*ins, pairs[t])
        got = torch.autograd.grad(out, ins + [mu, grav], grad_outputs=[torch.where(fluid, q, 0 * q) for q in bar],
                                  allow_unused=True)
        bar = [q if q is not None else torch.zeros_like(x) for q in got[:3]]
        dmu, dg = dmu + got[3], dg + got[4]
    rows = _rows(pos, vel, x, v.detach(), v.detach())
    return {"pos": rows["pos"], "vel": rows["vel"], "mu": dmu.detach(), "grav": dg.detach()}


def exact(case: dict, seed: int):
    kind = case["kind"]
    if _count(case) * case.get("steps", 1) > (8_000_000 if kind in ("dam3d", "launchers") else 50_000_000):
        return None
    if kind == "dam2d":
        fluid, bo, grid, r = _dam2d(case)
        p = S.params_dambreak(fluid, bo, grid, r)
        pos = np.empty((_count(case), 4), np.float32)
        L.call("cmag_reference_initial_state", C.byref(p), pos.shape[0], pos.ctypes.data)
        lo = [float(p.clamp_lo[0]), float(p.clamp_lo[1])]
        pos, vel = _dam_state(torch.as_tensor(pos, device=DEV), _gen(seed), 2 * r, lo,
                              (fluid[0] * 2 * r, fluid[1] * 2 * r), 0.5, True)
        return _dam_exact(p, pos, vel, 1)
    if kind == "dam3d":
        p, pos, vel = _state(case, seed)
        return _dam_exact(p, pos, vel, case["steps"])
    if kind in ("channel", "peristalsis"):
        p, pos, vel = _state(case, seed)
        return _channel_exact([p], [pos.shape[0]], pos, vel, case["steps"])
    if kind == "batch":
        inst = _batch_state(case, seed)
        pos, vel = (torch.cat([q[a] for q in inst]) for a in (1, 2))
        return _channel_exact([q[0] for q in inst], [q[1].shape[0] for q in inst], pos, vel, case["steps"])
    if kind == "adjoint":
        return _adjoint_exact(case, seed)
    return _launchers_exact(case, seed)
