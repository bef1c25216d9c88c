"""Closest and any hit through the four-child records (lux_amd/csrc/wide.hpp)
against the restated host LBVH walk, bit for bit: record counts around their
edges, ray counts on both sides of each lanes-per-ray rule, and boxes and rays
where the byte boxes' conservative arithmetic could go wrong."""

import numpy as np
import pytest

import oracle
from lux_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from lux_amd import lbvh

    lbvh.init(0)
    return lbvh


def check(gpu, tris, rays, boxes=None):
    print("wide", len(tris), len(rays), flush=True)
    boxes = W.triangle_boxes(tris) if boxes is None else boxes
    exp = oracle.OracleBvh(boxes).trace_closest(tris, rays)
    bvh = gpu.build_gpu_lbvh(boxes)
    hits = gpu.intersect_gpu_bvh_stackless(bvh, tris, rays)
    assert np.array_equal(hits["primitive_id"], exp["ids"])
    assert np.array_equal(hits["t"].view(np.uint32), np.asarray(exp["t"], np.float32).view(np.uint32))
    assert np.array_equal(gpu.trace_any(bvh, tris, rays), (exp["ids"] >= 0).astype(np.uint8))


def some_rays(n, seed, spread=1.0, centre=0.5):
    """Random rays, a third of them along axes or in coordinate planes, some as
    segments and some with a negative t_min."""
    rng = np.random.default_rng(seed)
    r = W.rays(n, seed=seed)
    r[:, 0:3] = centre + spread * (r[:, 0:3] - 0.5)
    k = np.arange(n) % 6
    r[k == 0, 3:5] = 0.0
    r[k == 1, 4] = 0.0
    r[k == 2, 7] = spread * rng.random(int((k == 2).sum())).astype(np.float32)
    r[k == 3, 6] = -0.3 * spread
    return r


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6, 9, 33, 1024, 1025, 4100])
def test_wide_record_counts(gpu, n):
    check(gpu, W.soup(n, seed=n, edge=(0.05, 0.4)), some_rays(777, n))


@pytest.mark.parametrize("rays", [1, 5, 63, 65, (1 << 14) - 1, (1 << 14) + 1, (1 << 16) + 1, (1 << 17) + 1])
def test_wide_ray_counts(gpu, rays):
    check(gpu, W.soup(3000, seed=3, edge=(0.02, 0.1)), some_rays(rays, 5))


@pytest.mark.parametrize("rays", [500, 140000])
@pytest.mark.parametrize("case", ["far", "tiny", "huge", "flat", "ties", "planes"])
def test_wide_awkward_boxes(gpu, case, rays):
    tris = W.soup(2000, seed=11, edge=(0.02, 0.2))
    spread, centre = 1.0, 0.5
    if case == "far":  # many record frames smaller than the float spacing of their corner
        tris, centre = (tris + np.float32(3000.0)).astype(np.float32), 3000.5
    elif case == "tiny":
        tris, spread, centre = (tris * np.float32(1e-3)).astype(np.float32), 1e-3, 0.5e-3
        tris = (tris * np.float32(16)).astype(np.float32)
    elif case == "huge":  # faces beyond the byte frames' range: records without culling
        tris, spread, centre = (tris * np.float32(4e18)).astype(np.float32), 4e18, 2e18
    elif case == "flat":  # every triangle in one of four planes
        t = tris.reshape(-1, 3, 3)
        t[:, :, 1] = (np.arange(len(t)) % 4)[:, None] * np.float32(0.25)
        tris = np.ascontiguousarray(t.reshape(-1, 9))
    elif case == "ties":
        tris = np.concatenate([tris[:700], tris[:700], tris[:300]])
    r = some_rays(rays, 17, spread, centre)
    if case == "planes":  # origins on box faces, directions along them
        v = tris.reshape(-1, 3)
        r[:, 0:3] = v[np.arange(rays) % len(v)]
        r[:, 3:6] = np.eye(3, dtype=np.float32)[np.arange(rays) % 3]
    check(gpu, tris, r)


@pytest.mark.parametrize("rays", [300, 140000])
def test_wide_boxes_without_end(gpu, rays):
    """Some primitive boxes reach to infinity (their triangles stay as they are)."""
    tris = W.soup(600, seed=21, edge=(0.05, 0.3))
    boxes = W.triangle_boxes(tris)
    boxes[::7, 3:] = np.inf
    boxes[3::11, 0] = -np.inf
    check(gpu, tris, some_rays(rays, 23), boxes)


@pytest.mark.parametrize("rays", [300, 140000])
def test_wide_odd_rays(gpu, rays):
    """Long, short, infinite and NaN rays among ordinary ones."""
    tris = W.soup(900, seed=31, edge=(0.05, 0.3))
    r = some_rays(rays, 33)
    k = np.arange(rays) % 50
    r[k == 1, 3:6] *= np.float32(1e20)
    r[k == 2, 3:6] *= np.float32(1e-9)
    r[k == 3, 3] = np.inf
    r[k == 4, 0] = np.nan
    r[k == 5, 4] = np.nan
    r[k == 6, 3:6] = 0.0
    r[k == 7, 7] = -1.0
    r[k == 8, 0:3] = np.float32(1e30)
    check(gpu, tris, r)
