"""What a tune word launches (CPU)."""
import os
import re

from sph2s_final_amd import autotune

STEP = os.path.join(os.path.dirname(autotune.__file__), "csrc", "step.hip")


def test_launch_shapes():
    d = autotune.launch_shape(0)
    assert d == {"density": {"waves_per_block": 4, "groups_per_wave": 1, "blocks_per_cu": None},
                 "force": {"waves_per_block": 4, "groups_per_wave": 1, "blocks_per_cu": None}}
    d = autotune.launch_shape(0x4352)
    assert d["density"] == {"waves_per_block": 2, "groups_per_wave": 1, "blocks_per_cu": 4}
    assert d["force"] == {"waves_per_block": 6, "groups_per_wave": 1, "blocks_per_cu": 8}
    d = autotune.launch_shape(0x90000)
    assert (d["density"]["waves_per_block"], d["force"]["waves_per_block"]) == (2, 6)
    d = autotune.launch_shape(0x500000)
    assert (d["density"]["groups_per_wave"], d["force"]["groups_per_wave"]) == (2, 2)


def test_waves_are_the_kernels():
    table = re.search(r"kTileWaves\[\] = \{([^}]*)\}", open(STEP).read()).group(1)
    assert tuple(int(v) for v in table.split(",")) == autotune.WAVES

