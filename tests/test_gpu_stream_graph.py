"""Contacts that form while captured steps run change the cache decision in the
middle of a call, with replays queued: the steps are captured anew and the run
equals the eager one bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from cabanadem_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_decision_changes_under_replay(gpu_lib):
    # a lattice 10 um short of contact that contracts by 33 mm/s a neighbour:
    # it touches after about 300 steps, between two samples of the contacts
    wl = W.plain_packed(dims=(83, 81, 79))
    st = wl.state
    centre = st.x.mean(axis=0)
    st.rad[:] = 0.985e-3
    st.u[:] = -(0.033 / 1.98e-3) * (st.x - centre)
    wl.gravity = (0., 0., 0.)
    wl.rebuild_every = 4
    out = []
    for graph in (False, True):
        s = wl.system(mode=1)
        s.set_graph(graph)
        s.step(200)
        assert not s.streaming()
        s.step(700)
        assert s.streaming()
        s.step(50)
        out.append(s.download(fields=("x", "u", "omega", "force", "torque", "ss_cnt")))
        s.close()
    assert out[0].ss_cnt.mean() > 3
    for f in ("x", "u", "omega", "force", "torque", "ss_cnt"):
        assert np.array_equal(getattr(out[0], f), getattr(out[1], f)), f
