"""Launch windows that halt with further steps already queued: those steps must do
nothing.  A first step with more parents than the planes hold, before a step with few;
and a window that halts (at a log point) after the Inside list has grown in its middle,
where the steps behind are queued without waiting.  Against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle.oracle import Oracle
from score_amd import synth
from score_amd.growth import GrowthMachine, same_trajectory
from score_amd.synth import ParamsSpec

pytestmark = pytest.mark.gpu


def _same(o, g):
    assert same_trajectory(o.trajectory(), g.trajectory())
    assert np.array_equal(o.grainmap(), g.grainmap())
    for a, b in zip(o.counts(), g.counts()):
        assert np.array_equal(a, b)
    for lst in (0, 1):
        fo, fg = o.front(lst), g.front(lst)
        act = fo["activity"] != 0
        assert np.array_equal(fo["activity"], fg["activity"])
        for f in ("cell", "rxfrac", "rxg"):
            assert np.array_equal(fo[f][act], fg[f][act]), (lst, f)


@pytest.mark.parametrize("chunks", [(13, 9, 3, 1000), (1000,), (12, 1000), (11, 2, 1, 1, 1000)])
def test_first_step_with_too_many_parents(require_gpu, chunks):
    e, n = 64, 30000
    dom = synth.make_voronoi_domain(e, e, e, n_grains=1, n_nuclei=n, seed=3)
    i = np.random.default_rng(1).choice((e - 4) ** 3, n, replace=False)
    dom.rxg_site[:] = (i % 60 + 2) + e * (i // 60 % 60 + 2) + e * e * (i // 3600 + 2)
    o = Oracle(dom, ParamsSpec())
    with GrowthMachine(dom, ParamsSpec()) as g:
        for c in chunks:
            o.step(c), g.step(c)
            _same(o, g)
        nf = o.trajectory()["nfull_inside"] + o.trajectory()["nfull_border"]
        # the planes hold 65536 parents at first
        assert nf[13] > 65536 > nf[:13].max() and nf[14] < 1000


@pytest.mark.parametrize("at", [11, 12, 13, 14, 16])
def test_halt_after_the_inside_list_grew(require_gpu, monkeypatch, at):
    monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", "1")
    dom = synth.make_voronoi_domain(40, 38, 36, n_grains=1, n_nuclei=200, seed=3)
    o = Oracle(dom, ParamsSpec())
    o.solve_rxgrowth()
    to = o.trajectory()
    prm = ParamsSpec(grainlog_at=(float(to["xcells"][at]), 0.7 * dom.N))
    o = Oracle(dom, prm)
    with GrowthMachine(dom, prm) as g:
        for c in (1, 9, 9, 1000):
            o.step(c), g.step(c)
            _same(o, g)
        for a, b in zip(o.grainlog(), g.grainlog()):
            assert np.array_equal(a, b)
    # the list of 3456 slots doubles at steps 0 and 11 and 13
    nI = to["nslots_inside"]
    assert 3456 < nI[0] <= 6912 and nI[10] <= 6912 < nI[11] <= 13824 < nI[13]
