"""A particle that is not finite, or far outside the grid, leaves the others alone.

Sums of the particles it is no neighbour of (every particle, if its position is
not finite) against the FP64 oracle with the suite's bars: density 1e-5 relative,
acceleration 1e-5 of max |a|.
"""
import numpy as np
import pytest

import oracle as O
from sph2s_final_amd import FIELD_ACCEL, SPH_DEBUG_ACCEL, ParticleData, Solver, scenes

pytestmark = pytest.mark.gpu

TOL = 1e-5
H = float(scenes.dam_break((8, 8, 8), seed=1).config.h)


def _config():
    return scenes.dam_break((8, 8, 8), seed=1).config


def _gpu_step(cfg, pos, vel):
    """Densities and accelerations by particle, and the device error bits."""
    with Solver(ParticleData(len(pos), pos, vel), None, cfg) as s:
        s.set_debug(SPH_DEBUG_ACCEL)
        s.Advance(scenes.DT)
        bits = s.device_errors()
        order = np.argsort(s.ids())
        return s.densities()[order], s.download(FIELD_ACCEL)[order], bits


def _oracle_step(cfg, pos, vel):
    ref = O.step(O.params_from_config(cfg), pos, vel, scenes.DT)
    rho, acc = np.empty_like(ref["rho"]), np.empty_like(ref["acc"])
    rho[ref["perm"]], acc[ref["perm"]] = ref["rho"], ref["acc"]
    return rho, acc


def _assert_close(rho, acc, want_rho, want_acc):
    assert np.max(np.abs(rho - want_rho) / want_rho) <= TOL
    assert np.max(np.abs(acc - want_acc)) <= TOL * np.max(np.abs(want_acc))


@pytest.mark.parametrize("bad", [(np.nan, 0, 0), (-np.nan, 0, 0), (0, np.nan, 0), (0, 0, np.nan),
                                 (np.inf, 0, 0), (-np.inf, 0, 0), (np.nan, np.nan, np.inf)])
def test_positions_that_are_not_finite(bad):
    # They share the boundary cells of finite particles: 254 in a cell at most,
    # so that the cells have x-bins.
    rng = np.random.default_rng(5)
    n, k = 1500, 12
    pos = rng.uniform(0.05 * H, 3.9 * H, size=(n + k, 3)).astype(np.float32)
    vel = rng.normal(0.0, 0.2, size=(n + k, 3)).astype(np.float32)
    bad = np.array(bad, np.float32)
    pos[n:] = np.where(bad == 0, pos[n:], bad)
    print(f"case positions {bad}", flush=True)
    rho, acc, _ = _gpu_step(_config(), pos, vel)
    _assert_close(rho[:n], acc[:n], *_oracle_step(_config(), pos[:n], vel[:n]))
