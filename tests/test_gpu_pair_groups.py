"""The neighbour walk of groups of 32 particles, where it can go wrong.

Group remainders (1 to 65 particles), a batch whose scenes end inside a group,
candidate lists from a few to several rings of four 60-candidate words, grid
cells smaller and larger than h, a group that spans rows or lies at both ends of
long ones, and particles outside the grid.  Each against the FP64 oracle with
the suite's bars: density 1e-5 relative, acceleration 1e-5 of max |a*|, for these
sums of at most a few hundred FP32 terms (FP64 partial sums in the density).
"""
import numpy as np
import pytest
import torch

import oracle as O
from sph2s_final_amd import (FIELD_ACCEL, FIELD_DENSITY, SPH_DEBUG_ACCEL, BatchSolver,
                             ParticleData, Solver, scenes)
from sph2s_final_amd._capi import SPH_FLAG_WALL_CLAMP

pytestmark = pytest.mark.gpu

TOL = 1e-5
H = float(scenes.dam_break((8, 8, 8), seed=1).config.h)


def _config(cells=1.0):
    """The 8^3 dam break's configuration with grid cells of h / cells."""
    cfg = scenes.dam_break((8, 8, 8), seed=1).config
    hi = [cfg.grid.origin[d] + cfg.grid.dims[d] * cfg.grid.spacing for d in range(3)]
    cfg.grid.spacing = float(np.float32(cfg.h / cells))
    for d in range(3):
        cfg.grid.dims[d] = int(np.ceil((hi[d] - cfg.grid.origin[d]) / cfg.grid.spacing))
    return cfg


def _state(n, seed, lo, hi):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(lo, hi, size=(n, 3)).astype(np.float32)
    return pos, rng.normal(0.0, 0.2, size=(n, 3)).astype(np.float32)


def _check(name, cfg, pos, vel):
    print(f"case {name}: n={len(pos)}", flush=True)
    with Solver(ParticleData(len(pos), pos, vel), None, cfg) as s:
        s.set_debug(SPH_DEBUG_ACCEL)
        s.Advance(scenes.DT)
        s.synchronize()
        assert s.device_errors() == 0
        rho, acc = s.densities(), s.download(FIELD_ACCEL)
    ref = O.step(O.params_from_config(cfg), pos, vel, scenes.DT)
    assert np.max(np.abs(rho - ref["rho"]) / ref["rho"]) <= TOL
    assert np.max(np.abs(acc - ref["acc"])) <= TOL * np.max(np.abs(ref["acc"]))


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 127, 129])
def test_group_remainders(n):
    _check("remainder", _config(), *_state(n, n, 1.2 * H, 3.1 * H))


@pytest.mark.parametrize("n", [3, 4, 5, 59, 60, 61, 119, 120, 121, 180, 181, 239, 241, 300])
def test_lists_around_the_words(n):
    # One cell again: a word holds 60 candidates, the ring four of them.
    _check("words", _config(), *_state(n, 1000 + n, 2.01 * H, 2.99 * H))


@pytest.mark.parametrize("n", [255, 256, 257, 319, 320, 321, 383, 511, 513, 640, 641, 769])
def test_lists_longer_than_the_ring(n):
    # All in one cell: every group's list holds all n.
    _check("one cell", _config(), *_state(n, n, 2.01 * H, 2.99 * H))


@pytest.mark.parametrize("cells", [0.4, 0.5, 1.0, 1.01, 2.0, 2.7, 4.0])
def test_grid_spacings(cells):
    _check(f"h / {cells}", _config(cells), *_state(1500, 17, 0.2 * H, 4.9 * H))


@pytest.mark.parametrize("seed", [1, 2])
def test_sparse_rows_and_outside_the_grid(seed):
    # Groups that span many rows; then a third of the particles outside the
    # grid on every side, where the boundary cells hold them.
    _check("sparse", _config(), *_state(200, seed, 0.0, 5.2 * H))
    pos, vel = _state(600, seed, -1.5 * H, 6.5 * H)
    cfg = _config()
    cfg.flags &= ~SPH_FLAG_WALL_CLAMP
    _check("outside", cfg, pos, vel)


@pytest.mark.parametrize("length", [99, 106, 240])
def test_long_rows(length):
    # Groups whose targets lie at both ends of neighbouring rows, 100 h and
    # more apart.
    cfg = _config()
    cfg.grid.dims[0] = length + 2
    cfg.domain_hi[0] = float(np.float32((length + 2) * H))
    _check("long rows", cfg, *_state(24 * length, length, [0.1 * H, 0.3 * H, 0.3 * H],
                                     [(length + 1) * H, 3.3 * H, 2.3 * H]))


@pytest.mark.parametrize("counts", [[1, 33, 32, 31, 65, 700], [40, 1, 1, 511]])
def test_batch_groups_restart_at_each_scene(counts):
    cfg = _config()
    states = [_state(n, 7 + i, 0.3 * H, 3.6 * H) for i, n in enumerate(counts)]
    with BatchSolver([cfg] * len(counts), [p for p, _ in states], [v for _, v in states]) as b:
        b.set_debug(SPH_DEBUG_ACCEL)
        b.Advance(scenes.DT)
        b.synchronize()
        rho, acc = b.download(FIELD_DENSITY), b.download(FIELD_ACCEL)
    at = 0
    for n, (p, v) in zip(counts, states):
        print(f"case scene of {n}", flush=True)
        ref = O.step(O.params_from_config(cfg), p, v, scenes.DT)
        r, a = rho[at:at + n], acc[at:at + n]
        at += n
        assert np.max(np.abs(r - ref["rho"]) / ref["rho"]) <= TOL
        assert np.max(np.abs(a - ref["acc"])) <= TOL * np.max(np.abs(ref["acc"]))


def test_adjoint_of_uneven_scenes():
    # The adjoint's groups: remainders, lists of several rings and rows of all
    # lengths, two steps, against the FP64 adjoint with its suite's bar of 1e-3
    # (the parameters' against the largest of the batch: a scene's own can
    # cancel to nothing).
    from sph2s_final_amd.autograd import Rollout
    cfg = _config()
    states = [_state(33, 3, 1.1 * H, 2.4 * H), _state(1, 4, H, 2.0 * H),
              _state(700, 5, 0.3 * H, 4.2 * H), _state(31, 6, 1.1 * H, 2.4 * H),
              _state(321, 8, 2.01 * H, 2.99 * H)]
    refs, seeds = [], []
    for p, v in states:
        target = np.roll(p, 1, axis=0).astype(np.float64)
        refs.append(O.rollout_loss_grad(O.params_from_config(cfg), p, v, scenes.DT, 2, target))
        seeds.append(2.0 * (refs[-1]["x_final"] - target) / (3.0 * len(p)))

    def dev(parts):
        return torch.from_numpy(np.ascontiguousarray(np.concatenate(parts), np.float32)).cuda()

    with Rollout([cfg] * len(states), [len(p) for p, _ in states], scenes.DT, 2, 1) as r:
        r.forward(dev([p for p, _ in states]), dev([v for _, v in states]))
        gp, gv, gk, gm = r.backward(dev(seeds))
        torch.cuda.synchronize()
        assert r.device_errors() == 0
        gp, gv = gp.cpu().numpy(), gv.cpu().numpy()
    at = 0
    for (p, _), ref in zip(states, refs):
        print(f"case adjoint of {len(p)}", flush=True)
        for got, want in ((gp, ref["g_pos0"]), (gv, ref["g_vel0"])):
            err = np.max(np.abs(got[at:at + len(p)] - want))
            assert err <= 1e-3 * np.max(np.abs(want))
        at += len(p)
    for got, name in ((gk, "g_stiffness"), (gm, "g_viscosity")):
        want = np.array([ref[name] for ref in refs])
        assert np.max(np.abs(got - want)) <= 1e-3 * np.max(np.abs(want))
