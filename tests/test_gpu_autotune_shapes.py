"""The autotuner's trials are of different configurations: where small systems
take eight lanes per particle, a force tile has no effect, and another tile size
is only tried with a launch grid (one lane per particle)."""
from __future__ import annotations

import numpy as np
import pytest

from cabanadem_amd import abi
from gpu_helpers import granular_box, make_system

pytestmark = pytest.mark.gpu


def test_tile_sizes_are_tried_where_they_exist(gpu_lib):
    st, w, lo, hi = granular_box(12, 11, 10, spacing_r=1.97, jitter_r=0.03, vsigma=0.05, seed=3)
    s = make_system(st, w, dt=1e-6, rc=2.3e-3, lo=lo, hi=hi, rebuild_every=20, skin=0.3e-3)
    s.step(20)
    before = s.download()
    r = s.autotune(trial_steps=40)
    seen = [tuple(t[k] for k in ("rebuild_every", "grid_blocks", "graph", "force_pass", "block", "tile_rows"))
            for t in r.trials()]
    assert len(seen) == len(set(seen))
    eight = [t for t in r.trials() if t["force_pass"] == abi.FORCE_PASS_FUSED and t["grid_blocks"] == 0]
    assert {t["block"] for t in eight} == {128}
    assert {t["block"] for t in r.trials()} == {64, 128, 256}
    after = s.download()
    for f in ("x", "u", "omega", "ss_cnt"):
        assert np.array_equal(getattr(before, f), getattr(after, f)), f
    s.close()
