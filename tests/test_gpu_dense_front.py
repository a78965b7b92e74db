"""Dense nuclei: fronts of more than 0.4 slots a cell, in lists that start with enough,
double beside the old one, take what room is left beside it, or go by way of host
memory; against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle.oracle import Oracle
from score_amd import abi, synth
from score_amd.growth import GrowthMachine, same_trajectory
from score_amd.synth import ParamsSpec

pytestmark = pytest.mark.gpu


def _same(dom, prm, least):
    o = Oracle(dom, prm)
    o.solve_rxgrowth()
    to = o.trajectory()
    assert to["nslots_inside"].max() > least * dom.N
    with GrowthMachine(dom, prm) as g:
        g.solve_rxgrowth()
        assert same_trajectory(to, g.trajectory())
        assert np.array_equal(o.grainmap(), g.grainmap())
        for a, b in zip(o.counts(), g.counts()):
            assert np.array_equal(a, b)
        fo, fg = o.front(abi.LIST_INSIDE), g.front(abi.LIST_INSIDE)
        assert np.array_equal(fo["activity"], fg["activity"])


# the list starts with more than 2^20 slots from 5.3M cells on
@pytest.mark.parametrize("density,grains,least", [(3e-2, 2900, 0.5), (1e-2, 1, 0.6), (1e-3, 1, 0.25)])
def test_list_from_the_density(require_gpu, density, grains, least):
    dom = synth.make_voronoi_domain(185, 177, 179, n_grains=grains, n_nuclei=int(density * 185 * 177 * 179), seed=2)
    _same(dom, ParamsSpec(xmax=0.7), least)


@pytest.mark.parametrize("start", [0.07, 0.2, 0.3, 0.35, 0.4, 0.43])
@pytest.mark.parametrize("shape", [(60, 60, 60), (61, 57, 63)])
def test_list_grows_past_half(require_gpu, monkeypatch, start, shape):
    N = shape[0] * shape[1] * shape[2]
    monkeypatch.setenv("SCORE_GM_FRONT_SLOTS", str(int(start * N)))
    dom = synth.make_voronoi_domain(*shape, n_grains=108, n_nuclei=int(0.02 * N), seed=2)
    _same(dom, ParamsSpec(), 0.42)
