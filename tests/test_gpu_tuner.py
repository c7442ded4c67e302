"""The tuner times launch shapes, not words: walled scenes, whose passes have one
shape, keep word 0 with equal default and tuned times, and no two words of one shape
are compared (their difference would be noise)."""
import numpy as np
import pytest

from sph2s_final_amd import ParticleData, Solver, TwoScaleSolver, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tension", [0.0, 0.8])
def test_walled_scenes_have_one_shape(tension):
    sc = scenes.walled_tank_small()
    sc.config.tension = tension
    print(f"case tune walls tension={tension}", flush=True)
    with Solver(ParticleData(sc.n, sc.positions), ParticleData(len(sc.walls), sc.walls),
                sc.config) as s:
        s.Advance(sc.dt, 2)
        before = s.positions()
        word, ms = s.autotune(sc.dt, reps=2)
        assert word == 0 and ms[0] == ms[1] and ms[2] == ms[3] and ms[0] > 0 and ms[2] > 0
        assert np.array_equal(s.positions(), before)
        s.set_tune(0x4452)  # still a word


def _canonical(word):
    """Whether each field is the first that selects its shape."""
    force_waves, density_block, force_block = word >> 4 & 0xF, word >> 16 & 3, word >> 18 & 3
    return force_waves <= 5 and density_block in (0, 2) and force_block == 0


@pytest.mark.parametrize("n", [8, 24])
def test_words_of_one_shape_are_timed_once(n):
    sc = scenes.dam_break((n, n, n), seed=2)
    print(f"case tune {sc.n}", flush=True)
    with Solver(ParticleData(sc.n, sc.positions), None, sc.config) as s:
        for _ in range(4):
            s.Advance(sc.dt)
            word, ms = s.autotune(sc.dt, reps=1)
            assert _canonical(word), hex(word)
            assert ms[1] <= ms[0] and ms[3] <= ms[2]
    sc = scenes.two_scale_dam_break(n, seed=2)
    with TwoScaleSolver(sc.config, sc.region_lo, sc.region_hi, sc.positions) as t:
        t.apply_split_merge()
        t.Advance(sc.dt)
        words, _ = t.autotune(reps=1)
        assert all(_canonical(w) for w in words), [hex(w) for w in words]
