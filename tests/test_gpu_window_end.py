"""The end of a launch window in its last commit pass: the largest weight kept while it
is below 1.0 (afterwards a pair's 1.0 is not reported any more), few and many blocks in
that pass, windows of one step and of many, against the oracle."""
import math

import numpy as np
import pytest

from oracle.oracle import Oracle
from score_amd import abi, synth
from score_amd.growth import GrowthMachine, same_trajectory
from score_amd.synth import ParamsSpec

pytestmark = pytest.mark.gpu


def _same(dom, prm, chunk):
    o, g = Oracle(dom, prm), GrowthMachine(dom, prm)
    while True:
        do, dg = o.step(chunk), g.step(chunk)
        assert do == dg
        if do:
            break
    assert same_trajectory(o.trajectory(), g.trajectory())
    assert np.array_equal(o.grainmap(), g.grainmap())
    pm = g.trajectory()["pmax"]
    g.close()
    return pm


@pytest.mark.parametrize("chunk", [1, 9, 1000])
def test_first_weight_of_one_inside_the_run(require_gpu, chunk):
    """Nuclei a few degrees off the grain they lie in: every weight is below 1.0 until
    the front meets a second grain."""
    dom = synth.make_voronoi_domain(40, 37, 33, n_grains=6, n_nuclei=12, seed=5)
    grid = dom.cellgrid.reshape(33, 37, 40)
    g0 = int(grid[16, 18, 20])
    q = dom.ori_quat[dom.defg_ori[g0]]
    a = math.radians(4.0)
    r = np.array([math.cos(a), math.sin(a), 0.0, 0.0])
    p = np.array([q[0] * r[0] - q[1] * r[1], q[0] * r[1] + q[1] * r[0], q[2] * r[0] + q[3] * r[1], q[3] * r[0] - q[2] * r[1]])
    dom.ori_quat[dom.rxg_ori] = p
    deep = grid == g0
    for ax in range(3):
        for sh in (-1, 1, -1, 1):
            deep = deep & np.roll(deep, sh, axis=ax)
    cells = np.nonzero(deep.ravel())[0]
    dom.rxg_site[:] = cells[np.linspace(0, len(cells) - 1, dom.n_rxg).astype(int)]
    pm = _same(dom, ParamsSpec(xmax=0.9), chunk)
    assert pm[0] < 1.0 and pm[-1] == 1.0


@pytest.mark.parametrize("nuclei", [1, 63, 64, 65, 5000])
@pytest.mark.parametrize("model", [abi.MOB_ROLLETTHOLM, abi.MOB_SEBALDGOTTSTEIN])
def test_blocks_of_the_last_pass(require_gpu, nuclei, model):
    e = 70 if nuclei == 5000 else 36
    dom = synth.make_voronoi_domain(e + 5, e + 2, e - 1, n_grains=9, n_nuclei=nuclei, seed=nuclei)
    _same(dom, ParamsSpec(mobility_model=model, xmax=0.3 if nuclei == 1 else 0.99), 7)


def test_one_step_windows_of_a_long_front(require_gpu):
    """Windows of one step whose compaction adds up more than 256 blocks' counts, and
    new pairs beyond and below the number one block resolves."""
    dom = synth.make_voronoi_domain(150, 140, 130, n_grains=6000, n_nuclei=9000, seed=4)
    prm = ParamsSpec(mobility_model=abi.MOB_SEBALDGOTTSTEIN, xmax=0.6)
    o, g = Oracle(dom, prm), GrowthMachine(dom, prm)
    o.solve_rxgrowth()
    g.solve_rxgrowth()
    to, tg = o.trajectory(), g.trajectory()
    assert same_trajectory(to, tg)
    assert np.array_equal(o.grainmap(), g.grainmap())
    assert (tg["nslots_inside"] + tg["nslots_border"]).max() > 256 * 2048
    assert tg["npending"].max() > 2048 and ((tg["npending"] > 0) & (tg["npending"] <= 2048)).any()
    g.close()


@pytest.mark.parametrize("nuclei", [64, 80000])
def test_first_step_beyond_the_parents_entries(require_gpu, nuclei):
    """More parents in the first step than there is room for at first (65536): the step
    is run again with its own propose pass."""
    dom = synth.make_voronoi_domain(64, 64, 64, n_grains=30, n_nuclei=nuclei, seed=3)
    # strictly interior sites, all different: the Border list has little room
    i = np.random.default_rng(1).choice(60 ** 3, nuclei, replace=False)
    dom.rxg_site[:] = (i % 60 + 2) + 64 * (i // 60 % 60 + 2) + 4096 * (i // 3600 + 2)
    prm = ParamsSpec(xmax=0.4 if nuclei > 64 else 0.9)
    o, g = Oracle(dom, prm), GrowthMachine(dom, prm)
    o.solve_rxgrowth()
    g.solve_rxgrowth()
    to, tg = o.trajectory(), g.trajectory()
    assert same_trajectory(to, tg)
    assert np.array_equal(o.grainmap(), g.grainmap())
    for a, b in zip(o.counts(), g.counts()):
        assert np.array_equal(a, b)
    assert (tg["nfull_inside"][0] + tg["nfull_border"][0] > 65536) == (nuclei == 80000)
    g.close()
