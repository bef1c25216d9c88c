"""Closest and any hit of instanced scenes through the four-child records of
both levels (lux_amd/csrc/two_level.hpp) against the restated preorder walk, bit
for bit: one-triangle meshes and one-instance scenes, instances in the same
place (every hit an exact tie), rays along axes in world or object space, and
ray counts on both sides of each lanes-per-ray rule."""

import numpy as np
import pytest

import oracle
from lux_amd import lbvh, two_level as TL, workloads as W

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 5, 300]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    lbvh.init(0)


def rays_toward(n, seed, extent, m):
    """Rays from around the instances' cube at the instances, a third of them along
    axes or in coordinate planes, some as segments and some with a negative t_min."""
    rng = np.random.default_rng(seed)
    r = np.array(W.rays(n, seed=seed), np.float32)
    r[:, 0:3] = (rng.random((n, 3)) * 2.4 - 1.2) * extent
    at = m[rng.integers(0, len(m), n)] @ np.append(np.full(3, 0.5), 1.0)
    at = (at[:, :3] + 0.4 * (rng.random((n, 3)) - 0.5)).astype(np.float32)
    r[:, 3:6] = at - r[:, 0:3]
    k = np.arange(n) % 6
    r[k == 0, 0:2] = at[k == 0, 0:2]
    r[k == 1, 1] = at[k == 1, 1]
    r[k == 0, 3:5] = 0.0
    r[k == 1, 4] = 0.0
    r[k == 2, 7] = 0.7
    r[k == 3, 6] = -0.5
    return r


def check(n_inst, n_rays, seed, place="random", extent=2.0):
    print("two-level records", n_inst, n_rays, place, flush=True)
    tris = np.concatenate([W.soup(k, seed=seed + k, edge=(0.2, 0.6)) for k in SIZES]).astype(np.float32)
    off = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.int32)
    mesh, m = W.instances_random(n_inst, len(SIZES), seed, extent=extent)
    m = np.array(m, np.float32)
    if place == "ties":
        mesh[:] = mesh[0]
        m[:] = m[0]
    if place == "axes":  # moved only: world axes are object axes
        m[:, :3, :3] = np.eye(3, dtype=np.float32)
    rec = TL.make_instances(mesh, m, tris=tris, mesh_offsets=off)
    rays = rays_toward(n_rays, seed, extent, m)
    exp = oracle.OracleTwoLevel(tris, off, mesh, rec["world_to_object"], rec["world_bounds"]).trace(rays)
    s = TL.TwoLevelScene(tris, off, rec)
    hits = s.intersect(rays)
    assert np.array_equal(hits["primitive_id"], exp["prim"])
    for k in ("t", "u", "v"):
        assert np.array_equal(hits[k].view(np.uint32), np.asarray(exp[k], np.float32).view(np.uint32)), k
    assert np.array_equal(s.occluded(rays).astype(bool), exp["prim"] >= 0)
    if n_rays > 500:
        assert 0 < int((exp["prim"] >= 0).sum()) < n_rays
    s.close()


@pytest.mark.parametrize("n_inst", [1, 2, 3, 5, 64, 65])
def test_instance_counts(n_inst):
    check(n_inst, 3001, 10 + n_inst)


@pytest.mark.parametrize("n_rays", [1, 63, (1 << 14) + 1, (1 << 16) + 1, (1 << 17) + 1])
def test_ray_counts(n_rays):
    check(20, n_rays, 7)


@pytest.mark.parametrize("n_rays", [2001, 140001])
@pytest.mark.parametrize("place", ["ties", "axes"])
def test_ties_and_axes(place, n_rays):
    check(9, n_rays, 21, place)


@pytest.mark.parametrize("n_rays", [2001, 140001])
@pytest.mark.parametrize("extent", [1e-3, 100.0])
def test_far_and_close_instances(extent, n_rays):
    check(12, n_rays, 33, extent=extent)
