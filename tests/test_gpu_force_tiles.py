"""The one-lane-per-particle force kernels at every tile size: a launch grid of
at least the tile count keeps small systems on them (by default they take eight
lanes per particle).  A wave's new state leaves through the LDS that held its
contact ids, so the lists' lengths are ragged here: lanes with none beside lanes
with many, partial waves and tiles, and tiles of a persistent grid."""
from __future__ import annotations

import numpy as np
import pytest

from cabanadem_amd import abi
from cabanadem_amd import workloads as W
from gpu_helpers import granular_box, make_system

pytestmark = pytest.mark.gpu

FIELDS = ("x", "u", "omega", "force", "torque", "ss_idx", "ss_cnt", "ss_x", "ss_y", "ss_z",
          "sw_x", "sw_y", "sw_z")
FULL_GRID = 1 << 20  # one workgroup per tile


def same(ref, s, what):
    got = s.download()
    for f in FIELDS:
        assert np.array_equal(getattr(ref, f), getattr(got, f)), (what, f)


def ragged(dims, seed):
    """Large spheres among small ones: 0 to 20 and more contacts side by side."""
    rng = np.random.default_rng(seed)
    st, w, lo, hi = granular_box(*dims, spacing_r=2.0, jitter_r=0.05, vsigma=0.3, omega_sigma=30., seed=seed,
                                 wall_offset=0.99e-3)
    big = rng.choice(st.n, size=max(1, st.n // 60), replace=False)
    st.rad[big] = 1.9e-3
    st.m[big] *= 1.9 ** 3
    st.I[big] *= 1.9 ** 5
    return st, w, dict(dt=2e-7, rc=4.1e-3, lo=lo, hi=hi, gravity=(0.3, -0.2, -9.81), rebuild_every=6,
                       skin=0.3e-3, max_contacts=24)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 13, 1), (13, 10, 1), (13, 12, 11), (26, 25, 24)])
def test_tiles(gpu_lib, dims, mode):
    """64, 128 and 256 slots, lane walk and tile-spread pass, one workgroup per
    tile and a persistent grid, against the eight-lane pass."""
    st, w, kw = ragged(dims, seed=7)
    ref = make_system(st, w, mode=mode, **kw)
    variants = [(block, p, grid) for block in (64, 128, 256)
                for p in (abi.FORCE_PASS_FUSED, abi.FORCE_PASS_WAVE) for grid in (FULL_GRID, 3)]
    systems = []
    for block, p, grid in variants:
        s = make_system(st, w, mode=mode, **kw)
        s.set_shape(block, 0)
        s.set_force_pass(p)
        s.set_launch(grid)
        systems.append(s)
    for steps in (1, 29):
        ref.step(steps)
        want = ref.download()
        for v, s in zip(variants, systems):
            s.step(steps)
            same(want, s, v)
    if st.n > 1000:
        assert want.ss_cnt.max() > 8 and (want.ss_cnt == 0).any()
    for s in systems + [ref]:
        s.build_neighbors()
        s.compute_forces()
    want = ref.download()
    for v, s in zip(variants, systems):
        same(want, s, v)
        s.close()
    ref.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_ensemble_tiles(gpu_lib, mode):
    wl = W.ensemble(n_systems=6, seed=8, nmin=150, nmax=2500, spacing_r=1.9, vsigma=0.5,
                    wall_offset=0.95 * 1.2e-3)
    ref = wl.system(mode=mode)
    ref.step(60)
    want = ref.download()
    assert want.ss_cnt.sum() > 0
    for block in (64, 128, 256):
        for p in (abi.FORCE_PASS_FUSED, abi.FORCE_PASS_WAVE):
            s = wl.system(mode=mode)
            s.set_shape(block, 0)
            s.set_force_pass(p)
            s.set_launch(FULL_GRID)
            s.step(60)
            same(want, s, (block, p))
            s.close()
    ref.close()


def test_automatic_cadence(gpu_lib):
    """The displacement check inside the lane walk at every tile size."""
    st, w, lo, hi = granular_box(10, 10, 10, spacing_r=2.05, jitter_r=0.02, vsigma=0.5, seed=23)
    kw = dict(dt=1e-6, rc=2.4e-3, lo=lo, hi=hi, gravity=(0., 0., -9.81), rebuild_every=abi.REBUILD_AUTO,
              skin=0.4e-3)
    ref = make_system(st, w, **kw)
    ref.step(500)
    want, c0 = ref.download(), ref.counters()
    assert c0.rebuilds >= 2 and c0.displacement_checks > c0.rebuilds
    for block in (64, 128, 256):
        s = make_system(st, w, **kw)
        s.set_shape(block, 0)
        s.set_launch(FULL_GRID)
        s.step(500)
        c = s.counters()
        assert (c.rebuilds, c.displacement_checks) == (c0.rebuilds, c0.displacement_checks)
        same(want, s, block)
        s.close()
    ref.close()
