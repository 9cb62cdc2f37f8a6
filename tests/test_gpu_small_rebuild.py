"""The one-workgroup rebuild that small systems take against the launch
sequence of larger ones (a binning grid of more than 8,192 cells keeps it):
the same cell order within a common grid cannot be forced from outside, so the
lists are compared as sets, and the runs against each other to rounding."""
from __future__ import annotations

import numpy as np
import pytest

from cabanadem_amd import abi
from cabanadem_amd import workloads as W
from gpu_helpers import granular_box, make_system, normwise, same_neighbor_sets

pytestmark = pytest.mark.gpu


def boxes(st, w, lo, hi, **kw):
    """The system binned in its own box (one workgroup) and in one with
    hundreds of empty cells along each side (the launch sequence)."""
    a = make_system(st, w, lo=lo, hi=hi, **kw)
    wide = 120 * kw["rc"]
    b = make_system(st, w, lo=np.asarray(lo) - wide, hi=np.asarray(hi) + wide, **kw)
    return a, b


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 1), (4, 4, 4), (9, 8, 7), (16, 16, 4), (25, 41, 1)])
@pytest.mark.parametrize("mode", [0, 1])
def test_small_rebuild(gpu_lib, dims, mode):
    """1 to 1,024 spheres (the limit) and 1,025, rebuilt every step."""
    st, w, lo, hi = granular_box(*dims, spacing_r=1.97, jitter_r=0.03, vsigma=0.3, omega_sigma=20., seed=4,
                                 wall_offset=0.99e-3)
    a, b = boxes(st, w, lo, hi, dt=1e-6, rc=2.4e-3, gravity=(0., 0., -9.81), mode=mode, rebuild_every=1)
    for s in (a, b):
        s.step(30)
        s.build_neighbors()
    assert same_neighbor_sets(a.neighbors(), b.neighbors())
    ga, gb = a.download(), b.download()
    # sums over contacts run in the two grids' slot orders: rounding
    for f in ("x", "u", "omega", "force", "torque"):
        assert normwise(getattr(ga, f), getattr(gb, f)) < 1e-9, f
    assert np.array_equal(ga.ss_cnt, gb.ss_cnt)
    a.close(), b.close()


def test_row_growth(gpu_lib):
    """Rows longer than the first capacity (48): the rebuild grows them and
    searches again from what the one-workgroup kernel left."""
    rng = np.random.default_rng(2)
    st, w, lo, hi = granular_box(9, 9, 9, spacing_r=2.05, jitter_r=0.02, vsigma=0.05, seed=6)
    st.x[:] = rng.uniform(0.2, 0.8, size=st.x.shape) * (hi - lo) + lo
    a, b = boxes(st, w, lo, hi, dt=1e-9, rc=5.5e-3, rebuild_every=1, max_contacts=32)
    for s in (a, b):
        s.build_neighbors()
    ca, cb = a.neighbors(max_n=729), b.neighbors(max_n=729)
    assert ca[0].max() > 48 and same_neighbor_sets(ca, cb)
    assert a.counters().max_neighbors_seen == ca[0].max() == b.counters().max_neighbors_seen
    a.close(), b.close()


def test_small_bonded_and_ensemble(gpu_lib):
    """Bonds, groups and an external force carried by the one-workgroup
    re-sort; several systems in one."""
    wl = W.bonded_block(dims=(7, 6, 5))
    rng = np.random.default_rng(1)
    wl.state.u[:] = rng.normal(0., 1e-2, size=wl.state.u.shape)
    out = []
    for wide in (0., 0.25):
        wl.lo = tuple(v - wide for v in wl.lo)
        wl.hi = tuple(v + wide for v in wl.hi)
        wl.rebuild_every = 3
        s = wl.system(mode=1)
        s.set_external_force(np.random.default_rng(2).normal(0, 1e-3, size=(wl.state.n, 3)))
        s.step(50)
        st, b = s.download(), s.download_bonds()
        out.append((st, b))
        s.close()
    (sa, ba), (sb, bb) = out
    assert normwise(sa.x, sb.x) < 1e-9 and normwise(sa.u, sb.u) < 1e-9
    assert np.array_equal(np.sort(ba.idx, axis=1), np.sort(bb.idx, axis=1))
    ens = W.ensemble(n_systems=3, seed=5, nmin=60, nmax=300, spacing_r=1.9, vsigma=0.5,
                     wall_offset=0.95 * 1.2e-3)
    ens.rebuild_every = 2
    s = ens.system()
    s.step(40)
    got = s.download(fields=("x", "u"))
    for k in range(3):
        one = ens.single(k)
        one.step(40)
        want = one.download(fields=("x", "u"))
        o = s.offsets
        assert np.array_equal(got.x[o[k]:o[k + 1]], want.x) and np.array_equal(got.u[o[k]:o[k + 1]], want.u)
        one.close()
    s.close()
