"""The map read between the steps changes nothing: it is assembled in the Inside list's
unused records, and the records a defragmentation leaves behind the list's end are in
use, since the next one may take them back."""
from __future__ import annotations

import numpy as np
import pytest

from oracle.oracle import Oracle
from score_amd import abi, synth
from score_amd.growth import GrowthMachine, same_trajectory
from score_amd.synth import ParamsSpec

pytestmark = pytest.mark.gpu


def _revival():
    """Two defragmentations with no completions between them, after the fast cells' end: the
    second takes 19,152 records back."""
    e = 38
    a = np.arange(2, e - 2, 3)
    dom = synth.make_voronoi_domain(e, e, e, n_grains=2, n_nuclei=len(a) ** 3, seed=3, rho_values=np.array([1e15, 1e14]))
    z, y, x = np.meshgrid(a, a, a, indexing="ij")
    dom.rxg_site[:] = (x + e * (y + e * z)).ravel()
    dom.rxg_ori[:] = dom.rxg_ori[0]
    dom.cellgrid = np.repeat(np.arange(e) >= 15, e * e).astype(np.uint32)
    return dom, ParamsSpec(xmax=5.0, defrag_at=(0.36 * dom.N,) * 2)


@pytest.mark.parametrize("encoding", [abi.MAP_CELLGRID, abi.MAP_RAW2GID])
def test_maps_between_defragmentations(require_gpu, encoding):
    dom, prm = _revival()
    o = Oracle(dom, prm)
    with GrowthMachine(dom, prm) as g:
        n = []
        for _ in range(45):
            o.step(1), g.step(1)
            assert np.array_equal(o.grainmap(encoding), g.grainmap(encoding))
            fo, fg = o.front(abi.LIST_INSIDE), g.front(abi.LIST_INSIDE)
            act = fo["activity"] != 0
            assert np.array_equal(fo["activity"], fg["activity"])
            for f in ("cell", "rxfrac", "rxg", "defg", "P"):
                assert np.array_equal(fo[f][act], fg[f][act]), f
            n.append(len(act))
        assert same_trajectory(o.trajectory(), g.trajectory())
        for a, b in zip(o.counts(), g.counts()):
            assert np.array_equal(a, b)
    # the list got shorter, then longer again without an infection
    t = o.trajectory()
    k = int(np.argmin(n[1:])) + 1
    assert n[k] < n[k - 1] and n[k + 1] - n[k] == 19152 and t["ninfected"][k + 1] == 0


@pytest.mark.parametrize("slots", [None, 1])
def test_maps_between_windows(require_gpu, monkeypatch, slots):
    if slots:
        monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", str(slots))
    dom = synth.make_voronoi_domain(34, 31, 29, n_grains=12, n_nuclei=400, seed=5)
    prm = ParamsSpec(defrag_at=(0.1 * dom.N, 0.3 * dom.N, 0.6 * dom.N))
    o = Oracle(dom, prm)
    with GrowthMachine(dom, prm) as g:
        done = False
        while not done:
            done = o.step(4)
            g.step(4)
            assert np.array_equal(o.grainmap(), g.grainmap())
        assert same_trajectory(o.trajectory(), g.trajectory())


def test_retired_cells_with_another_record(require_gpu):
    """A cell that is held twice and has retired once is its grain's in the map."""
    dom = synth.make_voronoi_domain(20, 28, 22, n_grains=1, n_nuclei=65, seed=38)
    prm = ParamsSpec(maxfill=0.045, xmax=0.7, defrag_at=(900.0, 1650.0, 5350.0, 5900.0, 6050.0, 8150.0, 8950.0))
    o = Oracle(dom, prm)
    o.solve_rxgrowth()
    fo = [o.front(lst) for lst in (abi.LIST_INSIDE, abi.LIST_BORDER)]
    held = np.concatenate([f["cell"][f["activity"] != 0] for f in fo])
    m = o.grainmap()
    assert (m[held] != abi.CURRENTLY_INFECTED).sum() > 100
    with GrowthMachine(dom, prm) as g:
        g.solve_rxgrowth()
        assert same_trajectory(o.trajectory(), g.trajectory())
        assert np.array_equal(m, g.grainmap())
