"""Device memory of a batch: what its passes read and write, and no more.

Per particle: state 32 bytes, density 4, acceleration 16, keys and permutation 12,
sort buffers 8, the internal order's state and packed factors 68, groups 0.5: 141; the
bar of 160 leaves room for the sort's tables and the allocator.
"""
import numpy as np
import pytest
import torch

from sph2s_final_amd import BatchSolver, scenes

pytestmark = pytest.mark.gpu


def test_bytes_per_particle():
    n = 1 << 20
    cfg = scenes.dam_break((8, 8, 8), seed=1).config
    pos = np.random.default_rng(1).uniform(0.0, 0.2, size=(n, 3)).astype(np.float32)
    print(f"case batch memory of {n}", flush=True)
    torch.cuda.init()
    BatchSolver([cfg], [pos[:64]]).close()
    free = torch.cuda.mem_get_info()[0]
    with BatchSolver([cfg], [pos]):
        used = free - torch.cuda.mem_get_info()[0]
    assert used <= 160 * n, used / n
