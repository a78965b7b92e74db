"""The infection passes with several regions where their partition and scans have
edges: steps of more parents than one round of the row scan takes (512 blocks of 64)
and just around one block, region grids of other shapes and of many regions (the
attempts into other regions' halos), against the oracle bit for bit."""
import numpy as np
import pytest

from score_amd import synth
from score_amd.synth import ParamsSpec

from oracle.oracle import Oracle
from test_gpu_regions import _gm, assert_final_equal_regions, region_domain

pytestmark = pytest.mark.gpu


def _same(dom, prm, T):
    print(f"regions T={T} {dom.nx}x{dom.ny}x{dom.nz} nuclei {dom.n_rxg}", flush=True)
    o, g = Oracle(dom, prm), _gm(dom, prm)
    o.solve_rxgrowth()
    g.solve_rxgrowth()
    assert_final_equal_regions(o, g, T)


@pytest.mark.parametrize("T", [5, 6, 12, 16, 27, 64])
def test_region_grids(require_gpu, T):
    _same(region_domain(T, seed=100 + T, n_grains=12, n_nuclei=20 + 4 * T), ParamsSpec(n_regions=T), T)


@pytest.mark.parametrize("T,nuclei", [(2, 63), (2, 64), (2, 65), (3, 130), (8, 513), (8, 40000), (4, 33000)])
def test_parents_at_block_edges(require_gpu, T, nuclei):
    """Every nucleus completes in the first step, so it has that many parents."""
    e = 24 if nuclei < 1000 else 72
    dom = synth.make_voronoi_domain(e, 2 * e, 2 * e - 1, n_grains=20, n_nuclei=nuclei, seed=T + nuclei)
    _same(dom, ParamsSpec(n_regions=T, xmax=0.5 if nuclei > 1000 else 0.99), T)


def test_long_front(require_gpu):
    """A front of more sweep blocks than compaction and propose pass share a launch for,
    on either side of the line within one run."""
    dom = synth.make_voronoi_domain(228, 216, 210, n_grains=600, n_nuclei=7700, seed=2)
    prm = ParamsSpec(n_regions=4, xmax=0.8)
    o, g = Oracle(dom, prm), _gm(dom, prm)
    o.solve_rxgrowth()
    g.solve_rxgrowth()
    tr = g.trajectory()
    slots = (tr["nslots_inside"] + tr["nslots_border"]).astype(np.int64)
    assert slots.min() * 3 // 2 < 1024 * 2048 < slots.max() * 3 // 2
    assert_final_equal_regions(o, g, 4)
