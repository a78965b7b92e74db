"""Domains of a batch, and of a served stream, that do not all fit into device memory at
the lengths their lists grow to: those that fail meanwhile are run again, and the
results are those of single runs."""
from __future__ import annotations

import gc

import numpy as np
import pytest

from score_amd import abi, synth
from score_amd.growth import GrowthMachine, Server, batch_run
from score_amd.synth import ParamsSpec

pytestmark = pytest.mark.gpu


def _domains(n):
    """Alike but for their nuclei's places, so that they grow in step."""
    return [synth.make_voronoi_domain(34, 31, 29, n_grains=1, n_nuclei=400, seed=3 + i) for i in range(n)]


def _single(dom):
    with GrowthMachine(dom) as g:
        r = g.solve_rxgrowth()
        return g.counts(), g.grainmap(), r


def _least_limit(monkeypatch, doms, hi=1 << 30):
    lo = 1
    while hi - lo > 4096:
        m = (lo + hi) // 2
        monkeypatch.setenv("SCORE_GM_MEM_LIMIT", str(m))
        try:
            for d in doms:
                _single(d)
            hi = m
        except abi.ScoreGmError as e:
            assert e.code == abi.ERR_OOM
            lo = m
    monkeypatch.delenv("SCORE_GM_MEM_LIMIT")
    return hi


@pytest.mark.parametrize("inflight", [2, 3, 8])
def test_batch_in_little_memory(require_gpu, monkeypatch, inflight):
    gc.collect()
    monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", "1")
    doms = _domains(8)
    want = [_single(d) for d in doms]
    least = _least_limit(monkeypatch, doms)
    for share in (1.0, 1.1, 1.5, 1.9, 1.98, 2.9, 2.97):
        print(f"inflight {inflight}, memory for {share} domains", flush=True)
        monkeypatch.setenv("SCORE_GM_MEM_LIMIT", str(int(least * share)))
        outs = batch_run(doms, ParamsSpec(), max_inflight=inflight, grainmaps=True)
        for (counts, gmap, r), o in zip(want, outs):
            assert np.array_equal(o["defg_counts"], counts[0]) and np.array_equal(o["rxg_counts"], counts[1])
            assert np.array_equal(o["grainmap"], gmap)
            assert o["result"]["step"] == r["step"] and o["result"]["t"] == r["t"]


def test_a_domain_that_never_fits(require_gpu, monkeypatch):
    """It is reported; the others are not."""
    gc.collect()
    monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", "1")
    doms = _domains(4)
    least = _least_limit(monkeypatch, doms)
    big = synth.make_voronoi_domain(70, 70, 70, n_grains=1, n_nuclei=4000, seed=9)
    monkeypatch.setenv("SCORE_GM_MEM_LIMIT", str(int(1.2 * least)))
    with Server(max_inflight=5) as srv:
        reqs = [srv.submit(d, ParamsSpec(), grainmap=True) for d in doms[:2] + [big] + doms[2:]]
        assert all(srv.wait(r, 60) for r in reqs)
    assert [r.outcome()["status"] for r in reqs] == [0, 0, abi.ERR_OOM, 0, 0]
