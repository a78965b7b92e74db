"""Grids and maps of 16 MiB and more cross the bus in 2 MiB chunks by several
threads: sizes just below, at and just above the line, with chunks left over, and a
last chunk of one row; both encodings, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle.oracle import Oracle
from score_amd import abi, synth
from score_amd.growth import GrowthMachine

pytestmark = pytest.mark.gpu

# 4 MiB cells is the line; 512 Ki cells are a chunk
SHAPES = [(127, 127, 260), (128, 128, 256), (129, 128, 254), (128, 128, 257), (161, 163, 171)]


@pytest.mark.parametrize("shape", SHAPES)
def test_grid_and_maps(require_gpu, shape):
    dom = synth.make_voronoi_domain(*shape, n_grains=50, n_nuclei=40, seed=shape[0])
    # every cell its own draw: a chunk in a wrong place would show
    dom.cellgrid = np.random.default_rng(shape[2]).integers(0, 50, dom.N).astype(np.uint32)
    with GrowthMachine(dom) as g, Oracle(dom) as o:
        for steps in (0, 2):
            if steps:
                o.step(steps), g.step(steps)
            for enc in (abi.MAP_CELLGRID, abi.MAP_RAW2GID):
                assert np.array_equal(o.grainmap(enc), g.grainmap(enc)), (steps, enc)
