"""Launch windows whose lists of completed cells are made at their start: shapes
at the edges of the bitmap's 16x8x8 bricks and of the 512-slot sweep chunks, runs
cut into chunks of steps, against the serial oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle.oracle import Oracle
from score_amd import abi, synth
from score_amd.growth import GrowthMachine, same_trajectory
from score_amd.synth import ParamsSpec

pytestmark = pytest.mark.gpu


def _same(dom, prm, chunks):
    o, g = Oracle(dom, prm), GrowthMachine(dom, prm)
    k = 0
    while True:
        n = chunks[k % len(chunks)]
        do, dg = o.step(n), g.step(n)
        assert do == dg, k
        for lst in (abi.LIST_INSIDE, abi.LIST_BORDER):
            fo, fg = o.front(lst), g.front(lst)
            for f in ("activity", "cell", "rxfrac", "rxg"):
                act = fo["activity"] != 0
                assert np.array_equal(fo["activity"], fg["activity"]), (k, lst, f)
                assert np.array_equal(fo[f][act], fg[f][act]), (k, lst, f)
        if do:
            break
        k += 1
    assert same_trajectory(o.trajectory(), g.trajectory())
    assert np.array_equal(o.grainmap(), g.grainmap())
    for a, b in zip(o.counts(), g.counts()):
        assert np.array_equal(a, b)
    g.close()


@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 3, 40), (16, 8, 8), (17, 9, 9), (15, 7, 7), (33, 16, 17), (32, 24, 5),
                                   (18, 10, 33), (49, 3, 16)])
def test_shapes_at_brick_edges(require_gpu, shape):
    nx, ny, nz = shape
    N = nx * ny * nz
    dom = synth.make_voronoi_domain(nx, ny, nz, n_grains=max(1, N // 300), n_nuclei=max(1, N // 200), seed=sum(shape))
    _same(dom, ParamsSpec(xmax=1.0), (9, 1, 4))


@pytest.mark.parametrize("maxfill,chunks", [(0.1, (9,)), (0.1, (8, 3)), (0.045, (16,))])
def test_recycled_slots_across_windows(require_gpu, maxfill, chunks):
    """Many nuclei, so that several sweep blocks hand out recycled slots in most
    steps and blocks further up are reached only late in a window."""
    dom = synth.make_voronoi_domain(45, 41, 38, n_grains=30, n_nuclei=900, seed=21)
    _same(dom, ParamsSpec(maxfill=maxfill), chunks)


def test_front_of_many_sweep_blocks(require_gpu):
    """A front beyond the 2^19 slots up to which no scan pass runs."""
    dom = synth.make_voronoi_domain(150, 140, 130, n_grains=200, n_nuclei=9000, seed=4)
    o, g = Oracle(dom, ParamsSpec()), GrowthMachine(dom, ParamsSpec())
    o.step(70)
    g.step(70)
    assert g.trajectory()["nslots_inside"].max() > 1 << 19
    assert same_trajectory(o.trajectory(), g.trajectory())
    fo, fg = o.front(abi.LIST_INSIDE), g.front(abi.LIST_INSIDE)
    act = fo["activity"] != 0
    for f in ("cell", "rxfrac", "rxg"):
        assert np.array_equal(fo[f][act], fg[f][act]), f
    assert np.array_equal(fo["activity"], fg["activity"])
    g.close()


@pytest.mark.parametrize("slots,chunks", [(1, (9,)), (1, (2, 5)), (3000, (9, 1))])
def test_inside_list_grows(require_gpu, monkeypatch, slots, chunks):
    """The Inside list starts short, so that it has to grow before a commit pass (in
    the first and in later steps of a window, twice in a row, and to a slot per cell
    by way of host memory), with later arrivals and defragmentation between."""
    monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", str(slots))
    dom = synth.make_voronoi_domain(34, 31, 29, n_grains=12, n_nuclei=400, seed=5)
    _same(dom, ParamsSpec(defrag_at=(0.3 * dom.N, 0.6 * dom.N)), chunks)
    sheet = synth.make_rolled_sheet_domain(48, 40, 16, n_grains=30, n_nuclei=600, arrival_steps=20, seed=3)
    _same(sheet, ParamsSpec(rh_hagb_m0=2.0), chunks)
