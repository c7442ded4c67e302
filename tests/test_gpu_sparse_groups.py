"""Groups of 32 particles spread over many cells and rows, which are scanned
directly, beside groups that are walked together.

Spray from one particle in 50 cells to 6 a cell, films across the rows (one row
per few particles), grid cells of h / 4 to 2.5 h, a pool with spray above it,
particles outside the grid, batches, the blended coupling and the adjoint.  Each
against the FP64 oracle with the suite's bars: density 1e-5 relative, acceleration
1e-5 of max |a*|, gradients 1e-3.
"""
import numpy as np
import pytest
import torch

import oracle as O
from sph2s_final_amd import (FIELD_ACCEL, FIELD_DENSITY, SPH2_COUPLING_BLENDED,
                             SPH2_SPLIT_REFERENCE, SPH_DEBUG_ACCEL, BatchSolver, scenes)
from sph2s_final_amd._capi import SPH_FLAG_WALL_CLAMP
from test_gpu_pair_groups import H, TOL, _check, _config, _state
from test_two_scale_blended import (_blended, _compare_step, _gpu, _oracle,
                                    _seed_oracle_from_gpu, _split_state)

pytestmark = pytest.mark.gpu


def _open(edge, cells=1.0):
    """The configuration with a domain and grid of that edge, in units of h."""
    cfg = _config(cells)
    for d in range(3):
        cfg.grid.dims[d] = int(np.ceil(edge * cells))
        cfg.domain_hi[d] = float(np.float32(edge * H))
    return cfg


@pytest.mark.parametrize("per_cell", [0.02, 0.2, 0.6, 1.0, 1.5, 3.0, 6.0])
@pytest.mark.parametrize("n", [33, 1500])
def test_spray(per_cell, n):
    edge = max(2.0, (n / per_cell) ** (1 / 3))
    _check(f"spray {per_cell}", _open(edge), *_state(n, n, 0.0, edge * H))


@pytest.mark.parametrize("cells", [0.4, 0.5, 1.01, 2.0, 2.7, 4.0])
@pytest.mark.parametrize("per_h3", [0.3, 1.0])
def test_spray_in_other_cells(cells, per_h3):
    edge = (800 / per_h3) ** (1 / 3)
    _check(f"spray in cells of h / {cells}", _open(edge, cells), *_state(800, 8, 0.0, edge * H))


@pytest.mark.parametrize("per_cell", [1, 4, 9, 12, 16])
@pytest.mark.parametrize("dx", [1, 2, 3, 40])
def test_films_across_rows(per_cell, dx):
    cfg = _open(12.0)
    cfg.grid.dims[0] = dx
    pos, vel = _state(144 * per_cell, per_cell, 0.0, 12.0 * H)
    pos[:, 0] *= np.float32(0.8 / 12.0)
    _check(f"film {per_cell} of {dx}", cfg, pos, vel)


def test_spray_above_a_pool_and_outside():
    pos, vel = _state(2400, 3, 0.0, 10.0 * H)
    pos[:2000, 1] *= np.float32(0.2)
    cfg = _open(10.0)
    _check("spray above a pool", cfg, pos, vel)
    cfg.tension = 0.8
    _check("with tension", cfg, pos, vel)
    cfg = _open(7.0)
    cfg.flags &= ~SPH_FLAG_WALL_CLAMP
    pos -= np.float32(1.5 * H)
    _check("outside", cfg, pos, vel)


def test_batch_of_spray():
    cfgs, states = [], []
    for i, (n, per_cell) in enumerate([(40, 0.05), (700, 0.5), (33, 8.0), (500, 2.0)]):
        edge = max(2.0, (n / per_cell) ** (1 / 3))
        cfgs.append(_open(edge))
        states.append(_state(n, 30 + i, 0.0, edge * H))
    with BatchSolver(cfgs, [p for p, _ in states], [v for _, v in states]) as b:
        b.set_debug(SPH_DEBUG_ACCEL)
        b.Advance(scenes.DT)
        b.synchronize()
        rho, acc = b.download(FIELD_DENSITY), b.download(FIELD_ACCEL)
    at = 0
    for cfg, (p, v) in zip(cfgs, states):
        print(f"case spray scene of {len(p)}", flush=True)
        ref = O.step(O.params_from_config(cfg), p, v, scenes.DT)
        r, a = rho[at:at + len(p)], acc[at:at + len(p)]
        at += len(p)
        assert np.max(np.abs(r - ref["rho"]) / ref["rho"]) <= TOL
        assert np.max(np.abs(a - ref["acc"])) <= TOL * np.max(np.abs(ref["acc"]))


@pytest.mark.parametrize("n", [60, 900])
@pytest.mark.parametrize("tension", [0.0, 0.8])
def test_blended_spray(n, tension):
    sc = scenes.two_scale_dam_break(24, seed=9)
    sc.config.tension = tension
    edge = float(sc.config.domain_hi[0])
    sc.positions, sc.velocities = _state(n, n, 0.01 * edge, 0.99 * edge)
    base = _split_state(sc)
    o = _oracle(sc)
    with _gpu(sc) as s:
        s.set_state(base.get(0, "pos").astype(np.float32), base.get(0, "vel").astype(np.float32),
                    base.get(0, "id"), base.get(1, "pos").astype(np.float32),
                    base.get(1, "vel").astype(np.float32), base.get(1, "id"), base.get(1, "tag"))
        s.set_options(coupling=SPH2_COUPLING_BLENDED, split_offsets=SPH2_SPLIT_REFERENCE,
                      blend_increment=0.25, velocity_cap=0.8)
        rng = np.random.default_rng(n)
        for r in (0, 1):
            s.set_blend(r, rng.uniform(0.1, 1.0, s.counts()[r]).astype(np.float32))
        _blended(o, split_offsets=SPH2_SPLIT_REFERENCE, blend_increment=0.25, velocity_cap=0.8)
        print(f"case blended spray n={n} counts={s.counts()[:2]} tension={tension}", flush=True)
        _seed_oracle_from_gpu(o, s)
        o.step(sc.dt)
        s.Advance(sc.dt)
        s.synchronize()
        _compare_step(s, o)


def test_adjoint_of_spray():
    from sph2s_final_amd.autograd import Rollout
    cfgs, states = [], []
    for i, (n, per_cell) in enumerate([(40, 0.5), (600, 1.0), (33, 8.0), (400, 3.0)]):
        edge = max(2.0, (n / per_cell) ** (1 / 3))
        cfgs.append(_open(edge))
        states.append(_state(n, 50 + i, 0.0, edge * H))
    refs, seeds = [], []
    for cfg, (p, v) in zip(cfgs, states):
        target = np.roll(p, 1, axis=0).astype(np.float64)
        refs.append(O.rollout_loss_grad(O.params_from_config(cfg), p, v, scenes.DT, 2, target))
        seeds.append(2.0 * (refs[-1]["x_final"] - target) / (3.0 * len(p)))

    def dev(parts):
        return torch.from_numpy(np.ascontiguousarray(np.concatenate(parts), np.float32)).cuda()

    with Rollout(cfgs, [len(p) for p, _ in states], scenes.DT, 2, 1) as r:
        r.forward(dev([p for p, _ in states]), dev([v for _, v in states]))
        gp, gv, gk, gm = r.backward(dev(seeds))
        torch.cuda.synchronize()
        assert r.device_errors() == 0
        gp, gv = gp.cpu().numpy(), gv.cpu().numpy()
    at = 0
    for (p, _), ref in zip(states, refs):
        print(f"case adjoint of spray of {len(p)}", flush=True)
        for got, want in ((gp, ref["g_pos0"]), (gv, ref["g_vel0"])):
            err = np.max(np.abs(got[at:at + len(p)] - want))
            assert err <= 1e-3 * np.max(np.abs(want))
        at += len(p)
    for got, name in ((gk, "g_stiffness"), (gm, "g_viscosity")):
        want = np.array([ref[name] for ref in refs])
        assert np.max(np.abs(got - want)) <= 1e-3 * np.max(np.abs(want))
