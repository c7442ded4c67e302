"""What a user of this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values.  ``prepare`` makes what a program holds
before the call (a solver or a rollout on the GPU, device arrays), ``run`` is
one pass through the public entry points, ``exact`` the same result in 64 bits
by plain torch and numpy, ``work`` what a pass cannot do without.

Kinds of cases:
  frame     a single-scale ``Solver`` advances one displayed frame (a few steps
            of 1 ms) of a sloshing pool, and the positions and velocities are
            read on the GPU by particle id, as a renderer or an analysis does.
            A pool under gravity settles at a density that grows with depth,
            rho = rho0 exp(g (surface - y) / k): the state that a dam break
            spends most of its run in.
  walls     the same with surface tension in a tank of boundary particles
            around a pillar (the reference scene's tank and constants).
  two_scale one displayed step of the two-scale solver (a refined corner of a
            pool), read with ``render_tensors``; ``blended`` selects the
            reference's own coupling.
  sweep     a parameter study: uneven, independent dam breaks run together for
            some steps from device arrays (``Rollout.forward``).
  gradient  the differentiable rollout: forward and backward, with the
            gradients of the initial state and of each scene's parameters.
  sort      the standalone stable sort of (key, value) pairs.
"""
from __future__ import annotations

import math
import random
from ctypes import c_uint32, c_void_p

import numpy as np
import torch

import sph2s_final_amd as sph
from sph2s_final_amd import scenes
from sph2s_final_amd.autograd import Rollout, rollout

GRAVITY = 9.81
PLASTIC = (0.8191725133961645, 0.6710436067037893, 0.5497004779019703)  # the R3 sequence


def listed():
    return [
        # A small interactive scene: one frame of 8 steps, launches count.
        {"name": "frame_4k", "kind": "frame", "nx": 16, "ny": 16, "nz": 16, "steps": 8},
        # The 32,768-particle dam break's size and domain, settled.
        {"name": "frame_32k", "kind": "frame", "nx": 32, "ny": 32, "nz": 32, "steps": 8},
        # A long, ragged channel.
        {"name": "frame_183k", "kind": "frame", "nx": 131, "ny": 37, "nz": 38, "steps": 4},
        # The 1,000,000-particle dam break's size and domain, settled: the largest.
        {"name": "frame_1m", "kind": "frame", "nx": 100, "ny": 100, "nz": 100, "steps": 4},
        # The reference scene's tank (860,390 wall particles), a layer of fluid in it.
        {"name": "walls_204k", "kind": "walls", "x1": 1.6, "z0": -0.1, "z1": 0.5, "depth": 0.09,
         "steps": 4},
        # Two scales, the 63^3 pool with its refined corner, one step a frame.
        {"name": "two_scale_250k", "kind": "two_scale", "n": 63, "blended": False},
        # The same under the reference's blended coupling, smaller.
        {"name": "two_scale_blended_64k", "kind": "two_scale", "n": 40, "blended": True},
        # A few small scenes together.
        {"name": "sweep_small", "kind": "sweep", "scenes": 5, "lo": 1500, "hi": 9000, "steps": 24},
        # Many uneven scenes together.
        {"name": "sweep_uneven", "kind": "sweep", "scenes": 24, "lo": 4096, "hi": 98304,
         "steps": 24},
        # Fitting the initial state and the parameters of a few scenes.
        {"name": "gradient_65k", "kind": "gradient", "scenes": 4, "nx": 32, "ny": 32, "nz": 16,
         "steps": 12, "every": 4},
        # The same at the size of the 16-scene fitting task, in fewer steps.
        {"name": "gradient_1m", "kind": "gradient", "scenes": 16, "nx": 64, "ny": 32, "nz": 32,
         "steps": 4, "every": 2},
        # The sort by itself, on keys of a 19-bit cell grid.
        {"name": "sort_1m", "kind": "sort", "n": 1_000_003, "bits": 19},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "walls", "two_scale", "two_scale",
                       "sweep", "sweep", "gradient", "gradient", "sort"])
    if kind == "frame":
        edge = _log(rng, 2000, 1_000_000) ** (1 / 3)
        a, b = _log(rng, 0.7, 1.5), _log(rng, 0.7, 1.5)
        nx, nz = max(8, round(edge * a)), max(8, round(edge * b))
        return {"kind": kind, "nx": nx, "nz": nz,
                "ny": max(8, min(round(edge / (a * b)), 1_000_000 // (nx * nz))),
                "steps": rng.randint(2, 4) if edge > 50 else rng.randint(4, 8)}
    if kind == "walls":
        return {"kind": kind, "x1": round(rng.uniform(0.2, 1.6), 3), "z0": -0.1,
                "z1": round(rng.uniform(0.0, 0.5), 3), "depth": round(rng.uniform(0.05, 0.09), 3),
                "steps": rng.randint(2, 4)}
    if kind == "two_scale":
        blended = rng.random() < 0.4
        return {"kind": kind, "n": round(_log(rng, 14, 40 if blended else 63)), "blended": blended}
    if kind == "sweep":
        lo = round(_log(rng, 1000, 8000))
        return {"kind": kind, "scenes": rng.randint(2, 20), "lo": lo,
                "hi": round(lo * _log(rng, 2, 10)), "steps": rng.randint(6, 24)}
    if kind == "gradient":
        edge = _log(rng, 2000, 60000) ** (1 / 3)
        steps = rng.randint(3, 8)
        return {"kind": kind, "scenes": rng.randint(1, 10), "nx": max(8, round(1.5 * edge)),
                "ny": max(8, round(edge)), "nz": max(8, round(edge / 1.5)), "steps": steps,
                "every": rng.randint(2, steps)}
    return {"kind": kind, "n": round(_log(rng, 2000, 1_000_000)),
            "bits": rng.choice([12, 17, 19, 21, 24])}


# ---- inputs ------------------------------------------------------------------

def _pool(boxes, extent, h_eq, stiffness, seed, speed):
    """Particles of a settled pool over the floor of the box `extent` (h_eq:
    the depth it would have at rest density), so many over each part
    (n, x0, x1, z0, z1) of the floor, and a sloshing velocity field."""
    rng = np.random.Generator(np.random.PCG64(seed))
    lx, _, lz = extent
    a = GRAVITY / stiffness
    depth = np.log1p(a * h_eq) / a
    parts = []
    for n, x0, x1, z0, z1 in boxes:
        u = np.mod(np.arange(1, n + 1, dtype=np.float64)[:, None] * np.array(PLASTIC)
                   + rng.random(3), 1.0)
        p = np.empty((n, 3))
        p[:, 0] = x0 + u[:, 0] * (x1 - x0)
        p[:, 1] = depth - np.log1p(a * h_eq * u[:, 1]) / a
        p[:, 2] = z0 + u[:, 2] * (z1 - z0)
        p += rng.normal(0.0, 0.1 * scenes.SPACING, p.shape)
        p[:, 0] = np.clip(p[:, 0], x0 + 1e-4, x1 - 1e-4)
        p[:, 1] = np.maximum(p[:, 1], 1e-4)
        p[:, 2] = np.clip(p[:, 2], z0 + 1e-4, z1 - 1e-4)
        parts.append(p)
    pos = np.concatenate(parts)
    ph = rng.uniform(0.5, 1.0, 2) * speed
    vel = rng.normal(0.0, 0.1 * speed, pos.shape)
    vel[:, 0] += ph[0] * np.sin(math.pi * pos[:, 0] / lx)
    vel[:, 1] -= ph[0] * np.cos(math.pi * pos[:, 0] / lx) * pos[:, 1] * math.pi / lx
    vel[:, 2] += ph[1] * np.sin(2 * math.pi * pos[:, 2] / lz)
    return pos.astype(np.float32), vel.astype(np.float32)


def _frame_inputs(case, seed, boxes=None):
    n = case["nx"] * case["ny"] * case["nz"]
    ext = [case[a] / scenes.REFERENCE_LATTICE for a in ("nx", "ny", "nz")]
    cfg = sph.SolverConfiguration.FromConstants(
        scenes.H, scenes.particle_mass(), scenes.REST_DENSITY, scenes.STIFFNESS, scenes.VISCOSITY,
        (0.0, 0.0, 0.0), ext)
    pos, vel = _pool(boxes or [(n, 0.0, ext[0], 0.0, ext[2])], ext,
                     n * scenes.SPACING ** 3 / (ext[0] * ext[2]), scenes.STIFFNESS, seed, 0.3)
    return cfg, pos, vel


def _wall_inputs(case, seed):
    spacing = 0.0075
    sc = scenes.walled_dam_break(fluid_lo=(0.0, 0.0, 0.0), fluid_hi=(0.1, 0.1, 0.1))
    grid = sph.Grid.MakeGrid((0.5 * spacing, 0.5 * spacing, case["z0"] + 0.5 * spacing),
                             (case["x1"], case["depth"], case["z1"]), spacing)
    pos = sph.ParticleData.CreateParticleBox(grid).host_positions()
    gap = 0.05  # the pillar and its shell of five layers
    clear = ((pos[:, 0] < 0.7 - gap) | (pos[:, 0] > 0.75 + gap)
             | (pos[:, 2] < 0.22 - gap) | (pos[:, 2] > 0.25 + gap))
    pos = np.ascontiguousarray(pos[clear])
    rng = np.random.Generator(np.random.PCG64(seed))
    pos += rng.uniform(-0.02 * spacing, 0.02 * spacing, pos.shape).astype(np.float32)
    vel = rng.normal(0.0, 0.02, pos.shape).astype(np.float32)
    cfg = sph.SolverConfiguration.MakeConfiguration(
        (-0.1, -0.1, -0.2), (1.7, 1.6, 0.6), pos.shape[0] * spacing ** 3, pos.shape[0], 35, 1000.0,
        30.0, 5.0, 88.1472, 0.8)
    return cfg, pos, vel, sc.walls


def _two_scale_inputs(case, seed):
    """A pool of n^3 particles with one corner refined: a fifth of it, kept
    2 mm off the corner's faces at first."""
    n, edge = case["n"] ** 3, case["n"] / scenes.REFERENCE_LATTICE
    x, z, gap = 0.6 * edge, 0.5 * edge, 2e-3
    boxes = [(n - 2 * (n // 5), 0.0, x - gap, 0.0, edge), (n // 5, x, edge, 0.0, z - gap),
             (n // 5, x + gap, edge, z + gap, edge)]
    cfg, pos, vel = _frame_inputs({"nx": case["n"], "ny": case["n"], "nz": case["n"]}, seed, boxes)
    return cfg, pos, vel, (x, 0.0, z), (edge, edge, edge)


def _batch_inputs(case, seed):
    rng = random.Random(seed)
    out, k, mu = [], [], []
    for s in range(case["scenes"]):
        if case["kind"] == "sweep":
            n = round(_log(random.Random(977 * s + case["scenes"]), case["lo"], case["hi"]))
            out.append(scenes.truncated_dam_break(n, 1000 * seed + s, velocity_sigma=0.05))
        else:
            out.append(scenes.dam_break((case["nx"], case["ny"], case["nz"]), 1000 * seed + s,
                                        velocity_sigma=0.05))
        k.append(rng.uniform(1.0, 5.0))
        mu.append(rng.uniform(1.0, 8.0))
    pos = torch.from_numpy(np.concatenate([s.positions for s in out])).cuda()
    vel = torch.from_numpy(np.concatenate([s.velocities for s in out])).cuda()
    return out, pos, vel, torch.tensor(k, dtype=torch.float32), torch.tensor(mu, dtype=torch.float32)


def _residual(pos, seed):
    """dL/dx of a fit whose target has spread further (stiffer), with noise."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    noise = torch.randn(pos.shape, generator=gen, device="cuda")
    return pos.detach() - 0.3 + 0.05 * noise


class _DeviceArray:
    """A borrowed device array, for torch.as_tensor."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False),
                                         "version": 2}


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "steps": case.get("steps", 1)}
    if kind in ("frame", "walls"):
        if kind == "frame":
            cfg, pos, vel = _frame_inputs(case, seed)
            walls = None
        else:
            cfg, pos, vel, w = _wall_inputs(case, seed)
            walls = sph.ParticleData(w.shape[0], w)
        n = pos.shape[0]
        st["solver"] = sph.Solver(sph.ParticleData(n, pos, vel), walls, cfg)
        st["stream"] = torch.cuda.ExternalStream(st["solver"].views().stream)
        st["pos"] = torch.empty((n, 3), device="cuda")
        st["vel"] = torch.empty((n, 3), device="cuda")
    elif kind == "two_scale":
        cfg, pos, vel, lo, hi = _two_scale_inputs(case, seed)
        st["solver"] = sph.TwoScaleSolver(cfg, lo, hi, pos, vel)
        if case["blended"]:
            st["solver"].set_options(coupling=sph.SPH2_COUPLING_BLENDED,
                                     split_offsets=sph.SPH2_SPLIT_REFERENCE, velocity_cap=0.8)
        st["solver"].apply_split_merge()
        st["solver"].synchronize()
    elif kind in ("sweep", "gradient"):
        scs, pos, vel, k, mu = _batch_inputs(case, seed)
        st.update(pos=pos, vel=vel, k=k, mu=mu)
        st["rollout"] = Rollout([s.config for s in scs], [s.n for s in scs], scs[0].dt,
                                case["steps"], case.get("every", 20))
        if kind == "gradient":
            st["residual"] = _residual(pos, seed)
            for name in ("pos", "vel", "k", "mu"):
                st[name].requires_grad_(True)
    else:
        n, bits = case["n"], case["bits"]
        gen = torch.Generator(device="cuda").manual_seed(seed)
        # Cell hashes of particles that moved a little since they were last sorted.
        keys = torch.sort(torch.randint(0, 1 << bits, (n,), generator=gen, device="cuda"))[0]
        keys += torch.randint(-1, 2, (n,), generator=gen, device="cuda")
        st["keys"] = keys.clamp_(0, (1 << bits) - 1).to(torch.int32)
        st["vals"] = torch.randint(0, 1 << 31, (n,), generator=gen, device="cuda").to(torch.int32)
        st["out"] = (torch.empty_like(st["keys"]), torch.empty_like(st["vals"]))
        st["bits"] = bits
        st["bytes"] = int(sph.lib().sph_radix_sort_temp_bytes(n))
        st["temp"] = torch.empty(st["bytes"], dtype=torch.uint8, device="cuda")
    return st


# ---- one pass ----------------------------------------------------------------

def run(st):
    kind = st["kind"]
    if kind in ("frame", "walls"):
        s, stream = st["solver"], st["stream"]
        stream.wait_stream(torch.cuda.current_stream())
        s.Advance(scenes.DT, st["steps"])
        v = s.views()
        with torch.cuda.stream(stream):
            pos = torch.as_tensor(_DeviceArray(v.pos4, (v.n, 4)), device="cuda")
            vel = torch.as_tensor(_DeviceArray(v.vel4, (v.n, 4)), device="cuda")
            ids = pos.view(torch.int32)[:, 3].long()
            st["pos"].index_copy_(0, ids, pos[:, :3])
            st["vel"].index_copy_(0, ids, vel[:, :3])
        torch.cuda.current_stream().wait_stream(stream)
        return {"pos": st["pos"], "vel": st["vel"]}
    if kind == "two_scale":
        s = st["solver"]
        s.Advance(scenes.DT, 1)
        low, high = s.render_tensors(0), s.render_tensors(1)
        return {"low": low[0], "low_state": low[2], "high": high[0], "high_state": high[2]}
    if kind == "sweep":
        return {"pos": st["rollout"].forward(st["pos"], st["vel"], st["k"], st["mu"])}
    if kind == "gradient":
        for name in ("pos", "vel", "k", "mu"):
            st[name].grad = None
        x = rollout(st["rollout"], st["pos"], st["vel"], st["k"], st["mu"])
        x.backward(st["residual"])
        return {"pos": x.detach(), "grad_pos": st["pos"].grad, "grad_vel": st["vel"].grad,
                "grad_k": st["k"].grad, "grad_mu": st["mu"].grad}
    ko, vo = st["out"]
    rc = sph.lib().sph_radix_sort_pairs(
        c_void_p(st["keys"].data_ptr()), c_void_p(st["vals"].data_ptr()), c_void_p(ko.data_ptr()),
        c_void_p(vo.data_ptr()), c_uint32(ko.numel()), c_uint32(st["bits"]),
        c_void_p(st["temp"].data_ptr()), st["bytes"],
        c_void_p(torch.cuda.current_stream().cuda_stream))
    if rc != 0:
        raise RuntimeError(sph.lib().sph_last_error())
    return {"keys": ko, "vals": vo}


# ---- the work of a pass ------------------------------------------------------

LATTICE_NEIGHBOURS = 28          # within h = 2 spacings of a lattice point
PAIR_FLOPS = {"density": 12, "force": 30, "adjoint": 70}


def _pool_neighbours(h_eq, stiffness):
    """Mass-average neighbour count of a settled pool: rho grows linearly with the mass above."""
    return LATTICE_NEIGHBOURS * (1.0 + 0.5 * GRAVITY / stiffness * h_eq)


def work(case):
    kind = case["kind"]
    step = PAIR_FLOPS["density"] + PAIR_FLOPS["force"]
    if kind == "frame":
        n = case["nx"] * case["ny"] * case["nz"]
        h_eq = n * scenes.SPACING ** 3 * 32 * 32 / (case["nx"] * case["nz"])
        # state in and out once a step, positions and velocities by id once
        return {"bytes": 64.0 * n * case["steps"] + 56.0 * n,
                "flops": float(n) * case["steps"] * step * _pool_neighbours(h_eq, scenes.STIFFNESS)}
    if kind == "walls":
        n = case["x1"] * (case["z1"] - case["z0"]) * case["depth"] / 0.0075 ** 3
        return {"bytes": 64.0 * n * case["steps"] + 56.0 * n,
                "flops": n * case["steps"] * 35.0 * (step + 10)}
    if kind == "two_scale":
        low = case["n"] ** 3
        n = 0.8 * low + 8 * 0.2 * low
        h_eq = case["n"] * scenes.SPACING * (scenes.SPACING * 32) ** 2
        nb = _pool_neighbours(h_eq, scenes.STIFFNESS)
        return {"bytes": (64.0 + 16.0) * n, "flops": n * step * nb}
    if kind in ("sweep", "gradient"):
        if kind == "sweep":
            n = sum(round(_log(random.Random(977 * s + case["scenes"]), case["lo"], case["hi"]))
                    for s in range(case["scenes"]))
            return {"bytes": 64.0 * n * case["steps"] + 36.0 * n,
                    "flops": float(n) * case["steps"] * step * LATTICE_NEIGHBOURS}
        n = case["scenes"] * case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 64.0 * n * case["steps"] * 2 + 84.0 * n,
                "flops": float(n) * case["steps"] * LATTICE_NEIGHBOURS
                * (step + PAIR_FLOPS["adjoint"])}
    return {"bytes": 16.0 * case["n"], "flops": 0.0}


# ---- the same in 64 bits -----------------------------------------------------

def _pairs(xt, xs, h, chunk=1 << 17):
    """(i, j) of every pair with |xt_i - xs_j| < h, by a cell list of edge h."""
    lo = torch.minimum(xt.min(0).values, xs.min(0).values) - 2 * h
    ct, cs = ((xt - lo) / h).long(), ((xs - lo) / h).long()
    d = torch.maximum(ct.max(0).values, cs.max(0).values) + 3
    key, order = torch.sort((cs[:, 2] * d[1] + cs[:, 1]) * d[0] + cs[:, 0])
    xo = xs[order]
    got_i, got_j = [], []
    for a in range(0, xt.shape[0], chunk):
        c, x = ct[a:a + chunk], xt[a:a + chunk]
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                row = ((c[:, 2] + dz) * d[1] + c[:, 1] + dy) * d[0] + c[:, 0]
                b = torch.searchsorted(key, row - 1)
                cnt = torch.searchsorted(key, row + 1, right=True) - b
                i = torch.repeat_interleave(torch.arange(x.shape[0], device=x.device), cnt)
                first = torch.cumsum(cnt, 0) - cnt
                j = torch.arange(i.shape[0], device=x.device) - first[i] + b[i]
                near = ((x[i] - xo[j]) ** 2).sum(1) < h * h
                got_i.append(i[near] + a)
                got_j.append(order[j[near]])
    return torch.cat(got_i), torch.cat(got_j)


def _add(n, i, w):
    return torch.zeros((n, *w.shape[1:]), dtype=w.dtype, device=w.device).index_add(0, i, w)


def _c6(h):
    return 315.0 / (64.0 * math.pi * h ** 9)


def _c45(h):
    return 45.0 / (math.pi * h ** 6)


def _density(x, pairs, h, mass):
    i, j = pairs
    r2 = ((x[i] - x[j]) ** 2).sum(1)
    return mass * _c6(h) * _add(x.shape[0], i, (h * h - r2) ** 3)  # the pairs hold i = j too


def _accel(x, v, rho, pairs, h, mass, k, mu, tension, rest, gravity):
    i, j = pairs
    far = (x[i] != x[j]).any(1)
    i, j = i[far], j[far]
    d = x[i] - x[j]
    r2 = (d * d).sum(1)
    r = r2.sqrt()
    aa = k * (rho - rest) / rho ** 2
    f = ((aa[i] + aa[j]) * (h - r) ** 2 / r * mass * _c45(h))[:, None] * d
    f = f + (mu * mass * _c45(h) * (h - r) / (rho[i] * rho[j]))[:, None] * (v[j] - v[i])
    if tension:
        f = f - (tension * mass * _c6(h) * (h * h - r2) ** 3 / rho[i])[:, None] * d
    return _add(x.shape[0], i, f) + gravity


def _integrate(x, v, a, dt, cfg):
    v = v + dt * a
    x = x + dt * v
    if cfg.flags & sph.SPH_FLAG_WALL_CLAMP:
        lo = x.new_tensor(list(cfg.domain_lo))
        hi = x.new_tensor(list(cfg.domain_hi))
        out = (x < lo) | (x > hi)
        v = torch.where(out, -cfg.restitution * v, v)
        x = torch.where(x < lo, lo, torch.where(x > hi, hi, x))
    return x, v


def _wall_accel(x, walls, cfg):
    i, j = _pairs(x, walls, cfg.h)
    d = x[i] - walls[j]
    r = (d * d).sum(1).sqrt()
    q = 2.0 * r / cfg.h
    b = torch.where(q < 2.0 / 3.0, torch.full_like(q, 2.0 / 3.0),
                    torch.where(q < 1.0, 2.0 * q - 1.5 * q * q, 0.5 * (2.0 - q) ** 2))
    w = 0.02 * cfg.speed_sound ** 2 / r * b * cfg.boundary_mass / (cfg.mass + cfg.boundary_mass) / r
    return _add(x.shape[0], i, w[:, None] * d)


def _step(x, v, cfg, dt, k, mu, walls=None):
    xd = x.detach()
    pairs = _pairs(xd, xd, cfg.h)
    rho = _density(x, pairs, cfg.h, cfg.mass)
    g = x.new_tensor(list(cfg.gravity))
    a = _accel(x, v, rho, pairs, cfg.h, cfg.mass, k, mu, cfg.tension, cfg.rest_density, g)
    if walls is not None:
        a = a + _wall_accel(x, walls, cfg)
    return _integrate(x, v, a, dt, cfg)


def _cuda64(a):
    return torch.as_tensor(a).to("cuda", torch.float64)


def _exact_batch(case, seed):
    scs, pos, vel, k, mu = _batch_inputs(case, seed)
    grad = case["kind"] == "gradient"
    want = _residual(pos, seed).double() if grad else None
    dt = float(np.float32(scenes.DT))
    got = {n: [] for n in (("pos", "grad_pos", "grad_vel", "grad_k", "grad_mu") if grad else ("pos",))}
    at = 0
    for s, sc in enumerate(scs):
        x0, v0 = pos[at:at + sc.n].double(), vel[at:at + sc.n].double()
        ks, ms = (_cuda64(t[s:s + 1]) for t in (k, mu))
        leaves = [t.detach().clone().requires_grad_(grad) for t in (x0, v0, ks, ms)]
        with torch.set_grad_enabled(grad):
            x, v = leaves[0], leaves[1]
            for _ in range(case["steps"]):
                x, v = _step(x, v, sc.config, dt, leaves[2], leaves[3])
        got["pos"].append(x.detach())
        if grad:
            x.backward(want[at:at + sc.n])
            for n, t in zip(("grad_pos", "grad_vel", "grad_k", "grad_mu"), leaves):
                got[n].append(t.grad)
        at += sc.n
    return {n: torch.cat(t) for n, t in got.items()}


def _hash32(pos, edge, dims):
    """The reference's cell hash in 32 bits, for grids from the origin."""
    c = [np.clip((pos[:, d] / np.float32(edge)).astype(np.int32), 0, dims[d] - 1).astype(np.int64)
         for d in range(3)]
    return c[0] + dims[0] * (c[1] + dims[1] * c[2])


def _exact_two_scale(case, seed):
    """One step of the fixed coupling from the split state."""
    cfg, pos, vel, lo, hi = _two_scale_inputs(case, seed)
    lo, hi = np.float32(lo), np.float32(hi)
    h0, m0 = cfg.h, cfg.mass
    h1, m1 = 0.5 * h0, m0 / 8.0
    child = np.float32(h1 / 4.0)
    signs = np.array([[1.0 if (c >> d) & 1 else -1.0 for d in range(3)] for c in range(8)], np.float32)
    inside = ((pos >= lo) & (pos <= hi)).all(1)
    px = {0: pos[~inside], 1: (pos[inside][:, None, :] + child * signs).reshape(-1, 3)}
    pv = {0: vel[~inside], 1: np.repeat(vel[inside], 8, axis=0)}
    ext = [np.float32(cfg.domain_hi[d]) for d in range(3)]
    h, m, x, v, rho, acc = {0: h0, 1: h1}, {0: m0, 1: m1}, {}, {}, {}, {}
    for s in (0, 1):
        dims = [int(np.ceil(e / np.float32(h[s]))) for e in ext]
        order = np.argsort(_hash32(px[s], h[s], dims), kind="stable")
        x[s], v[s] = _cuda64(px[s][order]), _cuda64(pv[s][order])
    own = {s: _pairs(x[s], x[s], h[s]) for s in (0, 1)}
    cross = {s: _pairs(x[s], x[1 - s], h0) for s in (0, 1)}

    def near(s):
        i, j = cross[s]
        d = x[s][i] - x[1 - s][j]
        r2 = (d * d).sum(1)
        w = 0.5 * (_c6(h0) * (h0 * h0 - r2) ** 3 + _c6(h1) * (h1 * h1 - r2).clamp(min=0) ** 3)
        return i, j, d, r2.sqrt(), w

    for s in (0, 1):
        i, _, _, _, w = near(s)
        rho[s] = _density(x[s], own[s], h[s], m[s]) + m[1 - s] * _add(x[s].shape[0], i, w)
    k, mu, rest = cfg.stiffness, cfg.viscosity, cfg.rest_density
    for s in (0, 1):
        i, j, d, r, w = near(s)
        aa = {q: k * (rho[q] - rest) / rho[q] ** 2 for q in (0, 1)}
        p0, p1 = h0 - r, (h1 - r).clamp(min=0)
        g = 0.5 * (_c45(h0) * p0 ** 2 + _c45(h1) * p1 ** 2) / r
        l = 0.5 * (_c45(h0) * p0 + _c45(h1) * p1)
        f = m[1 - s] * ((aa[s][i] + aa[1 - s][j]) * g)[:, None] * d
        f = f + m[1 - s] * mu * (l / (rho[s][i] * rho[1 - s][j]))[:, None] * (v[1 - s][j] - v[s][i])
        acc[s] = _add(x[s].shape[0], i, f) + _accel(
            x[s], v[s], rho[s], own[s], h[s], m[s], k, mu, 0.0, rest, x[s].new_tensor(list(cfg.gravity)))
    dt = float(np.float32(scenes.DT))
    for s in (0, 1):
        x[s], v[s] = _integrate(x[s], v[s], acc[s], dt, cfg)
    new = ((x[0] >= _cuda64(lo)) & (x[0] <= _cuda64(hi))).all(1)
    kids = (x[0][new][:, None, :] + float(child) * _cuda64(signs)).reshape(-1, 3)
    return {"low": x[0][~new], "low_state": None, "high": torch.cat([x[1], kids]), "high_state": None}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("frame", "walls"):
        if kind == "frame":
            (cfg, pos, vel), walls = _frame_inputs(case, seed), None
        else:
            cfg, pos, vel, walls = _wall_inputs(case, seed)
            walls = _cuda64(walls)
        x, v = _cuda64(pos), _cuda64(vel)
        for _ in range(case["steps"]):
            x, v = _step(x, v, cfg, float(np.float32(scenes.DT)), cfg.stiffness, cfg.viscosity, walls)
        return {"pos": x, "vel": v}
    if kind == "two_scale":
        return None if case["blended"] else _exact_two_scale(case, seed)
    if kind in ("sweep", "gradient"):
        return _exact_batch(case, seed)
    return None  # whole numbers
