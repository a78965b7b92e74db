"""The pinned buffers of the staged copies are made for the workers of that moment: a
process that may use more processors afterwards reads its maps with as many workers."""
from __future__ import annotations

import os

import numpy as np
import pytest

from score_amd import abi, synth
from score_amd.growth import GrowthMachine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("few", [1, 4, 6])
def test_more_processors_after_creation(require_gpu, few):
    dom = synth.make_voronoi_domain(161, 163, 171, n_grains=50, n_nuclei=40, seed=few)
    dom.cellgrid = np.random.default_rng(few).integers(0, 50, dom.N).astype(np.uint32)
    cpus = os.sched_getaffinity(0)
    try:
        os.sched_setaffinity(0, set(sorted(cpus)[:few]))
        g = GrowthMachine(dom)
    finally:
        os.sched_setaffinity(0, cpus)
    with g:
        m = g.grainmap()
    placed = m != dom.cellgrid
    # only the nuclei's cells differ (INFECTED)
    assert placed.sum() == len(np.unique(dom.rxg_site)) and (m[placed] == abi.CURRENTLY_INFECTED).all()
