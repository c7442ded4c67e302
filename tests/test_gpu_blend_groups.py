"""The blended coupling's own-set passes at group remainders: sets whose counts
are no multiple of 32, groups over several rows, with and without tension, and
random blend weights, against the FP64 oracle with its suite's bars (density and
acceleration 1e-5, and the rest of _compare_step's).
"""
import numpy as np
import pytest

from sph2s_final_amd import SPH2_COUPLING_BLENDED, SPH2_SPLIT_REFERENCE, scenes
from test_two_scale_blended import (_blended, _compare_step, _gpu, _oracle,
                                    _seed_oracle_from_gpu, _split_state)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 7, 9, 12])
@pytest.mark.parametrize("tension", [0.0, 0.8])
def test_blended_groups(n, tension):
    sc = scenes.two_scale_dam_break(n, seed=20 + n)
    sc.config.tension = tension
    base = _split_state(sc, scenes.gaussian_velocities(sc.n, 0.3, n))
    o = _oracle(sc)
    with _gpu(sc) as s:
        s.set_state(base.get(0, "pos").astype(np.float32), base.get(0, "vel").astype(np.float32),
                    base.get(0, "id"), base.get(1, "pos").astype(np.float32),
                    base.get(1, "vel").astype(np.float32), base.get(1, "id"), base.get(1, "tag"))
        s.set_options(coupling=SPH2_COUPLING_BLENDED, split_offsets=SPH2_SPLIT_REFERENCE,
                      blend_increment=0.25, velocity_cap=0.8)
        rng = np.random.default_rng(n)
        for r in (0, 1):
            s.set_blend(r, rng.random(s.counts()[r]).astype(np.float32))
        _blended(o, split_offsets=SPH2_SPLIT_REFERENCE, blend_increment=0.25, velocity_cap=0.8)
        print(f"case blended groups n={sc.n} counts={s.counts()[:2]} tension={tension}", flush=True)
        _seed_oracle_from_gpu(o, s)
        o.step(sc.dt)
        s.Advance(sc.dt)
        s.synchronize()
        _compare_step(s, o)
