"""Materials changed between calls reach captured steps: dem_set_system_params on
a context of one system equals the same change on eager steps, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_helpers import granular_box, make_system

pytestmark = pytest.mark.gpu


def test_materials_reach_captured_steps(gpu_lib):
    st, w, lo, hi = granular_box(9, 8, 7, spacing_r=1.97, jitter_r=0.03, vsigma=0.3, seed=4, wall_offset=0.99e-3)
    out = []
    for graph, change in ((False, True), (True, True), (False, False)):
        s = make_system(st, w, dt=1e-6, rc=2.3e-3, lo=lo, hi=hi, rebuild_every=4, skin=0.3e-3)
        s.set_graph(graph)
        s.step(24)
        if change:
            s.set_system_params(0, cor_pp=0.5, cor_pw=0.6, friction_pp=0.7, friction_pw=0.1)
        s.step(24)
        out.append(s.download())
        s.close()
    eager, captured, unchanged = out
    for f in ("x", "u", "omega", "force", "torque"):
        assert np.array_equal(getattr(eager, f), getattr(captured, f)), f
    assert not np.array_equal(eager.u, unchanged.u)
