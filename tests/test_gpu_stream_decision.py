"""Whether a step's own streams go past the caches is decided from the state at
hand: known from the count and the bonds before the first step, from the contacts
within the first call, eager and captured, and again after another state is set.
Every kernel that goes past the caches gives the bits of the ones that do not
(steps that sample diagnostics never do)."""
from __future__ import annotations

import numpy as np
import pytest

from cabanadem_amd import abi
from cabanadem_amd import workloads as W

pytestmark = pytest.mark.gpu

FIELDS = ("x", "u", "omega", "force", "torque", "ss_cnt")
FUSED, WAVE = abi.FORCE_PASS_FUSED, abi.FORCE_PASS_WAVE


def state(s):
    st = s.download(fields=FIELDS)
    return {f: getattr(st, f) for f in FIELDS}


def assert_same(a, b, what):
    for f in FIELDS:
        assert np.array_equal(a[f], b[f]), (what, f)


def packed():
    return W.plain_packed(dims=(83, 81, 79))  # 531,000: decided by six contacts a sphere


@pytest.mark.parametrize("graph", [False, True])
def test_contacts_decide_in_the_first_call(gpu_lib, graph):
    wl = packed()
    s = wl.system(mode=1)
    s.set_graph(graph)
    s.set_params(rebuild_every=4)
    assert not s.streaming()  # no list yet
    s.step(40)
    assert s.streaming()
    # another state: the same lattice with spheres too small to touch
    far = wl.state.copy()
    far.rad[:] *= 0.9
    s.upload(far)
    s.step(40)
    assert not s.streaming()
    s.upload(wl.state)
    s.step(1)  # a call of one step: sampled behind its only pass
    assert s.streaming()
    # the other pass's limit lies lower
    s.upload(far)
    s.step(2)
    s.set_force_pass(WAVE)
    assert s.streaming() == (212. * wl.state.n > 0.7 * 256 * 2 ** 20)
    s.close()


def test_uploaded_contacts_decide_before_the_first_step(gpu_lib):
    wl = packed()
    a = wl.system(mode=1)
    a.step(2)
    st = a.download()
    a.close()
    b = wl.system(mode=1)
    assert not b.streaming()
    b.upload(st)
    assert b.streaming()
    b.close()


def test_count_and_bonds_decide_before_the_first_step(gpu_lib):
    for dims, on in (((60, 60, 60), False), ((111, 109, 107), True)):
        s = W.plain_large(dims=dims).system()
        assert s.streaming() == on
        s.step(3)
        assert s.streaming() == on
        s.close()
    wl = W.bonded_block(dims=(101, 61, 69))  # 425,000
    s = wl.system(mode=1)
    assert s.streaming()
    bonds = s.download_bonds()
    s.step(2)
    assert s.streaming()
    s.close()
    s = abi.System(wl.state.n, dt=wl.dt, cutoff=wl.cutoff, lo=wl.lo, hi=wl.hi, max_contacts=8, skin=wl.skin,
                   rebuild_every=wl.rebuild_every, physics_mode=1)
    s.upload(wl.state)
    s.enable_bonds(wl.max_bonds)
    assert not s.streaming()
    s.upload_bonds(bonds)
    assert s.streaming()
    s.close()


def run(wl, mode, steps, block=128, force_pass=FUSED, diag=0, graph=False):
    s = wl.system(mode=mode)
    s.set_shape(block, 0)
    s.set_force_pass(force_pass)
    s.set_diag_every(diag)
    s.set_graph(graph)
    for k in steps:
        s.step(k)
    out = state(s), s.streaming()
    s.close()
    return out


@pytest.mark.parametrize("bed,mode", [("loose", 0), ("packed", 1)])
def test_tiles_and_passes(gpu_lib, bed, mode):
    """Lane walk and tile-spread pass at 64, 128 and 256 slots past the limit."""
    wl = W.plain_large(dims=(111, 109, 107)) if bed == "loose" else packed()
    steps = (4, 22)  # across a rebuild
    want, _ = run(wl, mode, steps, diag=1)
    assert bed == "loose" or want["ss_cnt"].sum() > wl.state.n
    for block in (64, 128, 256):
        for p in (FUSED, WAVE):
            got, streaming = run(wl, mode, steps, block, p)
            assert streaming
            assert_same(want, got, (block, p))


def test_rebuild_past_the_caches(gpu_lib):
    """A count between the two passes' limits: everything through the caches in
    the lane walk, everything past them in the tile-spread pass."""
    wl = W.plain_large(dims=(101, 99, 103))
    want, streaming = run(wl, 0, (50,))
    assert not streaming
    got, streaming = run(wl, 0, (50,), force_pass=WAVE)
    assert streaming
    assert_same(want, got, "wave")


def test_captured_steps(gpu_lib):
    wl = packed()
    wl.rebuild_every = 3
    want, _ = run(wl, 1, (31, 20), diag=1)
    for graph in (False, True):
        got, streaming = run(wl, 1, (31, 20), graph=graph)
        assert streaming
        assert_same(want, got, graph)


def test_ensemble_tiles(gpu_lib):
    wl = W.ensemble(n_systems=70, seed=4, nmin=9000, nmax=20000, spacing_r=1.9, vsigma=0.5,
                    wall_offset=0.95 * 1.2e-3)
    want, _ = run(wl, 0, (4, 22), diag=1)
    assert want["ss_cnt"].sum() > 1000
    for block in (64, 256):
        got, streaming = run(wl, 0, (4, 22), block, WAVE)
        assert streaming
        assert_same(want, got, block)


def test_bonded(gpu_lib):
    wl = W.bonded_block(dims=(101, 61, 69))
    wl.state.u[:] = np.random.default_rng(3).normal(0., 1e-2, size=wl.state.u.shape)
    out = []
    for diag in (0, 1):
        s = wl.system(mode=1)
        s.set_diag_every(diag)
        s.step(30)
        assert s.streaming()
        out.append((state(s), s.download_bonds()))
        s.close()
    assert_same(out[0][0], out[1][0], "bonded")
    for h in out[0][1].HIST + ("idx", "init_len"):
        assert np.array_equal(getattr(out[0][1], h), getattr(out[1][1], h)), h
