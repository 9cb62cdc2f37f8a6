"""The eight-lanes-per-particle force pass that small systems take by default
against the one-lane kernel (a persistent launch grid keeps it): bit for bit
the same particle states and histories."""
from __future__ import annotations

import numpy as np
import pytest

from cabanadem_amd import abi
from cabanadem_amd import workloads as W
from gpu_helpers import granular_box, make_system

pytestmark = pytest.mark.gpu

FIELDS = ("x", "u", "omega", "force", "torque", "ss_idx", "ss_cnt", "ss_x", "ss_y", "ss_z",
          "sw_x", "sw_y", "sw_z")


def same(a, b):
    sa, sb = a.download(), b.download()
    for f in FIELDS:
        assert np.array_equal(getattr(sa, f), getattr(sb, f)), f
    return sa


def pair(make):
    """The same system twice: default launch, and a persistent grid."""
    a, b = make(), make()
    b.set_launch(24)
    return a, b


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("dims,cadence", [((1, 1, 1), 1), ((3, 5, 1), 1), ((7, 9, 11), 20), ((26, 27, 28), -1)])
def test_small_systems(gpu_lib, mode, dims, cadence):
    """One sphere, part of a workgroup, ragged sizes, just below the limit;
    spheres start on each other and on the walls."""
    st, w, lo, hi = granular_box(*dims, spacing_r=1.97, jitter_r=0.03, vsigma=0.3, omega_sigma=50., seed=3,
                                 wall_offset=0.99e-3)
    kw = dict(dt=1e-6, rc=2.3e-3, lo=lo, hi=hi, gravity=(0.3, -0.2, -9.81), mode=mode, rebuild_every=cadence,
              skin=0.3e-3)
    a, b = pair(lambda: make_system(st, w, **kw))
    for s in (a, b):
        s.step(40)
        s.set_external_force(np.random.default_rng(1).normal(0, 1e-4, size=(st.n, 3)))
        s.step(41)
        s.build_neighbors()
        s.compute_forces()
    got = same(a, b)
    if st.n > 100:
        assert got.ss_cnt.mean() > 1. and (got.sw_x != 0).any()
    a.close(), b.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_long_rows_and_lists(gpu_lib, mode):
    """Large spheres among small ones: rows beyond 16 neighbours and more than
    eight tracked contacts, moving and spinning walls, lists cut at
    max_contacts."""
    rng = np.random.default_rng(5)
    st, w, lo, hi = granular_box(14, 13, 12, spacing_r=1.9, jitter_r=0.05, vsigma=0.2, seed=9)
    big = rng.choice(st.n, size=40, replace=False)
    st.rad[big] = 1.9e-3
    st.m[big] *= 1.9 ** 3
    st.I[big] *= 1.9 ** 5
    walls = abi.Walls(w.x, w.normal, w.E, w.nu, w.G, u=rng.normal(0, 0.05, size=(w.n, 3)),
                      omega=rng.normal(0, 3., size=(w.n, 3)))
    a, b = pair(lambda: make_system(st, walls, dt=2e-7, rc=4.1e-3, lo=lo, hi=hi, mode=mode, rebuild_every=10,
                                    skin=0.3e-3, max_contacts=24))
    for s in (a, b):
        s.step(60)
    got = same(a, b)
    counts, _ = a.neighbors(max_n=128)
    assert got.ss_cnt.max() > 8 and counts.max() > 16
    a.close(), b.close()
    # more contacts than max_contacts: the same error on both paths
    errs = []
    for s in pair(lambda: make_system(st, walls, dt=2e-7, rc=4.1e-3, lo=lo, hi=hi, mode=mode, rebuild_every=10,
                                      skin=0.3e-3, max_contacts=4)):
        with pytest.raises(abi.DemError) as e:
            s.step(2)
        errs.append(str(e.value))
        s.close()
    assert errs[0] == errs[1] and "max_contacts" in errs[0]


@pytest.mark.parametrize("mode", [0, 1])
def test_small_ensemble(gpu_lib, mode):
    """Workgroups that straddle systems of different materials and walls."""
    wl = W.ensemble(n_systems=6, seed=8, nmin=150, nmax=2500, spacing_r=1.9, vsigma=0.5,
                    wall_offset=0.95 * 1.2e-3)
    assert wl.n <= 20000
    a, b = pair(lambda: wl.system(mode=mode))
    for s in (a, b):
        s.step(100)
    same(a, b)
    a.close(), b.close()
