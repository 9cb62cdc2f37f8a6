"""The step kernels that send their own streams past the caches once a step
outgrows them: bit for bit the results of the kernels that do not."""
from __future__ import annotations

import numpy as np
import pytest

from cabanadem_amd import workloads as W

pytestmark = pytest.mark.gpu


def state(s, fields):
    st = s.download(fields=fields)
    return {f: getattr(st, f) for f in fields}


@pytest.mark.parametrize("bed,dims,mode", [("loose", (111, 109, 107), 0), ("packed", (83, 81, 79), 1)])
def test_plain(gpu_lib, bed, dims, mode):
    """Sizes past the limit (a loose bed from 1.27M spheres; a packed one from
    its contacts, sampled at the end of the first call) against the split
    pass, whose kernels always go through the caches."""
    wl = W.plain_large(dims=dims) if bed == "loose" else W.plain_packed(dims=dims)
    f = ("x", "u", "omega", "force", "torque", "ss_cnt")
    out = []
    for split in (False, True):
        s = wl.system(mode=mode)
        s.set_force_pass(split)
        for _ in range(3):
            s.step(15)
        out.append(state(s, f))
        s.close()
    assert out[0]["ss_cnt"].sum() > 1000
    for k in f:
        assert np.array_equal(out[0][k], out[1][k]), k


def test_bonded(gpu_lib):
    """425,000 bonded spheres: one call keeps to the caches (no list has been
    sampled yet), two calls bypass them in the second."""
    wl = W.bonded_block(dims=(101, 61, 69))
    wl.state.u[:] = np.random.default_rng(3).normal(0., 1e-2, size=wl.state.u.shape)
    f = ("x", "u", "omega", "force", "torque")
    one, two = wl.system(mode=1), wl.system(mode=1)
    one.step(30)
    two.step(10)
    two.step(20)
    a, b = state(one, f), state(two, f)
    for k in f:
        assert np.array_equal(a[k], b[k]), k
    ba, bb = one.download_bonds(), two.download_bonds()
    for h in ba.HIST + ("idx", "init_len"):
        assert np.array_equal(getattr(ba, h), getattr(bb, h)), h
    one.close(), two.close()
