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


@pytest.mark.parametrize("n", [1, 63, 1023, 1025, 2047, 2048, 2049, 4096, 4097, 6144, 6145, 8193,
                               10239, 10240, 10241])
@pytest.mark.parametrize("bits", [1, 11, 20, 32])
def test_sorts_of_few_pairs(n, bits):
    # Around each block-sort size and the line to the general sort: a stable
    # sort, against numpy's.
    import ctypes

    import torch

    import sph2s_final_amd as sph
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint64).astype(np.uint32)
    keys[n // 2:] = keys[n // 2:] & np.uint32((1 << max(bits // 2, 1)) - 1)
    vals = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in (keys, vals)]
    out = [torch.empty_like(d) for d in dev]
    size = int(sph.lib().sph_radix_sort_temp_bytes(n))
    temp = torch.empty(size, dtype=torch.uint8, device="cuda")
    print(f"case sort {n} pairs of {bits} bits", flush=True)
    rc = sph.lib().sph_radix_sort_pairs(
        *[ctypes.c_void_p(d.data_ptr()) for d in dev + out], ctypes.c_uint32(n),
        ctypes.c_uint32(bits), ctypes.c_void_p(temp.data_ptr()), size,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(out[0].cpu().numpy().view(np.uint32), keys[order])
    assert np.array_equal(out[1].cpu().numpy().view(np.uint32), vals[order])


def test_batched_hash_across_scene_borders():
    # Waves of the histogram pass that span scenes: 700 scenes of 1 to 40
    # particles and one too large for the block sort, against each scene's own
    # hashes and ranges.
    from sph2s_final_amd import BatchSolver
    rng = np.random.default_rng(6)
    base = scenes.dam_break((8, 8, 8), seed=1).config
    counts = list(rng.integers(1, 41, 700)) + [10300]
    states = [rng.uniform(0.0, 0.22, size=(int(n), 3)).astype(np.float32) for n in counts]
    print(f"case batched hash of {sum(counts)}", flush=True)
    with BatchSolver([base] * len(counts), states) as b:
        b.Advance(scenes.DT)
        b.synchronize()
        assert b.device_errors() == 0
        got = b.download(FIELD_SORTED_HASH)
        cells = b.cell_offsets
        parts = b.part_offsets
    p = O.params_from_config(base)
    for s in list(range(0, 700, 7)) + [700]:
        keys = np.sort(O.hash_positions(p, states[s]), kind="stable")
        assert np.array_equal(got[parts[s]:parts[s + 1]] - np.uint32(cells[s]), keys)
