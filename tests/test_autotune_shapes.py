"""What a tune word launches, and cached words of an earlier meaning (CPU)."""
import json
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


class _FakeSolver:
    def __init__(self):
        self.tuned, self.set = 0, []

    def autotune(self, dt, reps):
        self.tuned += 1
        return 0x11, [1.0, 0.9, 2.0, 1.5]

    def set_tune(self, w):
        self.set.append(w)


def test_words_of_an_earlier_meaning_are_not_used(tmp_path):
    path = str(tmp_path / "tune.json")
    device = autotune._device_name()
    with open(path, "w") as f:
        json.dump({f"{device}|single|n=1000|cells=50|scenes=1": {"tune": 0x65, "ms": [1, 1, 1, 1]}}, f)
    s = _FakeSolver()
    r = autotune.tune(s, "single", 1000, 50, 1e-3, cache_path=path)
    assert not r["cached"] and r["tune"] == 0x11 and s.tuned == 1 and s.set == []
    assert r["launch"] == autotune.launch_shape(0x11)
    r = autotune.tune(s, "single", 1000, 50, 1e-3, cache_path=path)
    assert r["cached"] and r["tune"] == 0x11 and s.tuned == 1 and s.set == [0x11]
