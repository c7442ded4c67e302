"""Cell ranges and the order within cells, where runs of equal keys meet the
edges of the 256-slot blocks that find them and of the 64 keys looked at beyond.

Cells of chosen sizes one after the other along x, against the FP64 oracle:
hashes, permutation and cell ranges exact, density to 1e-5 (a particle out of
place or lost in a cell's order would change it by far more).
"""
import numpy as np
import pytest

import oracle as O
from sph2s_final_amd import (FIELD_CELL_END, FIELD_CELL_START, FIELD_SORTED_HASH,
                             FIELD_SORTED_INDEX, ParticleData, Solver, scenes)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [256, 1, 255, 2], [255, 257, 64, 192], [192, 65, 63, 64, 128], [1, 319, 320, 321],
    [128, 448, 500, 3], [576, 577, 1], [1, 1, 2100, 1], [200] * 6, [1] * 40,
])
def test_runs_at_block_edges(sizes):
    cfg = scenes.dam_break((8, 8, 8), seed=1).config
    h = float(cfg.h)
    per_row = 6
    rng = np.random.default_rng(sum(sizes) + len(sizes))
    parts = []
    for c, n in enumerate(sizes):
        cell = np.array([c % per_row, (c // per_row) % per_row, 2 * (c // per_row // per_row)])
        parts.append((cell + rng.uniform(0.05, 0.9, size=(n, 3))) * h)
    pos = rng.permutation(np.concatenate(parts)).astype(np.float32)
    cfg.grid.dims[0] = cfg.grid.dims[1] = cfg.grid.dims[2] = 8
    print(f"case runs {sizes}", flush=True)
    with Solver(ParticleData(len(pos), pos), None, cfg) as s:
        s.Advance(scenes.DT)
        s.synchronize()
        assert s.device_errors() == 0
        got = {f: s.download(f) for f in (FIELD_SORTED_HASH, FIELD_SORTED_INDEX, FIELD_CELL_START,
                                          FIELD_CELL_END)}
        rho = s.densities()
    ref = O.step(O.params_from_config(cfg), pos, np.zeros_like(pos), scenes.DT)
    assert np.array_equal(got[FIELD_SORTED_HASH], ref["hash"])
    assert np.array_equal(got[FIELD_SORTED_INDEX], ref["perm"])
    assert np.array_equal(got[FIELD_CELL_START], ref["cell_start"])
    assert np.array_equal(got[FIELD_CELL_END], ref["cell_end"])
    assert np.max(np.abs(rho - ref["rho"]) / ref["rho"]) <= 1e-5
