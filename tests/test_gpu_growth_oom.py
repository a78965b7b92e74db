"""Device memory that ends while the Inside list grows: beside the old list, and by way of
host memory, where the old list may be lost with it.  The handle reports it, takes no
further step and its read-backs answer or refuse."""
from __future__ import annotations

import gc

import pytest

from score_amd import abi, synth
from score_amd.growth import GrowthMachine
from score_amd.synth import ParamsSpec

pytestmark = pytest.mark.gpu


def _domain():
    return synth.make_voronoi_domain(34, 31, 29, n_grains=1, n_nuclei=400, seed=3)


def _reads(g):
    return [lambda: g.grainmap(), lambda: g.front(abi.LIST_INSIDE), lambda: g.front(abi.LIST_BORDER)]


def test_no_memory_for_the_list(require_gpu, monkeypatch):
    """No allocation succeeds any more from step s on."""
    monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", "1")
    dom = _domain()
    answered = refused = 0
    for s in range(0, 40):
        with GrowthMachine(dom, ParamsSpec()) as g:
            g.step(s)
            monkeypatch.setenv("SCORE_GM_MEM_LIMIT", "1")
            try:
                g.step(1000)
                err = None
            except abi.ScoreGmError as e:
                err = e
            monkeypatch.delenv("SCORE_GM_MEM_LIMIT")
            if err is None:
                continue
            assert err.code == abi.ERR_OOM
            with pytest.raises(abi.ScoreGmError) as again:
                g.step(1)
            assert again.value.code == abi.ERR_OOM
            codes = []
            for read in _reads(g):
                try:
                    read()
                    codes.append(0)
                except abi.ScoreGmError as e:
                    codes.append(e.code)
            # all of them or none
            assert codes in ([0] * 3, [abi.ERR_OOM] * 3), (s, codes)
            answered += codes[0] == 0
            refused += codes[0] != 0
    print("answered", answered, "refused", refused)
    assert answered and refused


def test_limit_must_be_a_number(require_gpu, monkeypatch):
    monkeypatch.setenv("SCORE_GM_MEM_LIMIT", "some")
    with pytest.raises(abi.ScoreGmError) as e:
        GrowthMachine(_domain())
    assert e.value.code == abi.ERR_ARG


def test_all_memory_is_given_back(require_gpu, monkeypatch):
    """The count of held bytes goes back to nothing with the handles."""
    monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", "1")
    gc.collect()
    dom = _domain()
    with GrowthMachine(dom) as g:
        g.solve_rxgrowth()
        g.grainmap(), g.counts(), g.front(abi.LIST_INSIDE)
    lo, hi = 1 << 10, 1 << 30
    # the least limit under which the run ends; it would creep up with bytes that stay counted
    need = []
    for _ in range(2):
        a, b = lo, hi
        while b - a > 4096:
            m = (a + b) // 2
            monkeypatch.setenv("SCORE_GM_MEM_LIMIT", str(m))
            try:
                with GrowthMachine(dom) as g:
                    g.solve_rxgrowth()
                b = m
            except abi.ScoreGmError as e:
                assert e.code == abi.ERR_OOM
                a = m
        need.append(b)
    assert need[0] == need[1] < hi
