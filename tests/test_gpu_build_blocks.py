"""Build and refit around the leaf-block counts where the threads per block of the
local pass change (lux_amd/csrc/lbvh.hip, launch_local): the node array against
the restated build, bit for bit."""

import numpy as np
import pytest

import oracle
from lux_amd import lbvh, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 1023, 1025, 96 * 1024, 96 * 1024 + 1, 384 * 1024, 384 * 1024 + 1])
def test_local_blocks(n):
    print("local blocks", n, flush=True)
    lbvh.init(0)
    tris = W.soup(n, seed=n, edge=(0.002, 0.02))
    boxes = W.triangle_boxes(tris)
    ids = np.arange(n, dtype=np.int32)
    bvh = lbvh.build_gpu_lbvh(boxes, ids)
    o = oracle.OracleBvh(boxes, ids)
    assert np.array_equal(bvh.nodes().view(np.uint32), o.nodes.view(np.uint32))
    moved = W.triangle_boxes(W.jitter(tris, sigma=2e-3, seed=1))
    assert lbvh.refit_gpu_lbvh(bvh, moved, ids)
    assert np.array_equal(bvh.nodes().view(np.uint32), o.refit(moved).nodes.view(np.uint32))
