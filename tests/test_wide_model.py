"""The walk over four-child records with byte boxes on the CPU: the library's own
header (lux_amd/csrc/wide.hpp) compiled with g++ over tests/simt, a wave's lanes as
fibers, against the oracle's right-first preorder walk; and trees whose arrays are
damaged, which must end in an error bit and never in an access out of range (each
such case runs in a process of its own, with indexes far outside the arrays)."""

import ctypes
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

import oracle
from conftest import load_golden
from lux_amd import workloads as W

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent
LIB = HERE / "_build" / "libwide_model.so"
WALK_ORDER, PRIM_RANGE = 2, 8  # DeviceError bits


@pytest.fixture(scope="session")
def model():
    import shutil

    include = Path("/opt/rocm/include")
    if not (include / "hip" / "hip_runtime_api.h").exists() or shutil.which("g++") is None:
        pytest.skip("needs g++ and the HIP headers")
    LIB.parent.mkdir(exist_ok=True)
    subprocess.run(["g++", "-std=c++20", "-O2", "-fPIC", "-shared", "-ffp-contract=off", f"-I{HERE / 'simt'}",
                    f"-I{ROOT / 'lux_amd' / 'csrc'}", f"-I{ROOT / 'include'}", f"-I{include}",
                    str(HERE / "wide_model.cpp"), "-o", str(LIB)], check=True)
    return WideModel


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


class WideModel:
    """Records over an oracle tree (as the library's build makes them)."""

    def __init__(self, tree, damage=None):
        self.lib = ctypes.CDLL(str(LIB))
        self.tree = tree
        n = self.n = tree.n
        self.nodes = np.ascontiguousarray(tree.nodes)
        self.left, self.right = tree.left.copy(), tree.right.copy()
        self.pre_internal = np.full(max(n - 1, 1), -1, np.int32)
        self.pre_leaf = np.full(n, -1, np.int32)
        esc = self.nodes["escape"]
        todo = [(0, 0)]  # (internal node, preorder position): the right child follows its parent
        while todo:
            i, k = todo.pop()
            self.pre_internal[i] = k
            for c, p in ((self.right[i], k + 1), (self.left[i], int(esc[k + 1]))):
                if c & 0x80000000:
                    self.pre_leaf[c & 0x7FFFFFFF] = p
                else:
                    todo.append((int(c), p))
        if damage:
            damage(self)
        self.wide = np.full((n - 1, 16), 0x7F7F7F7F, np.uint32)  # what the memory held
        self.wide_leaf = np.full(4 * (n - 1), 0x40000000, np.int32)
        self.fill_error = self.lib.wide_fill(n, _p(self.left), _p(self.right), _p(self.pre_internal),
                                             _p(self.pre_leaf), _p(self.nodes), _p(self.wide), _p(self.wide_leaf))

    def trace(self, tris, rays, any_hit=False, group=1):
        t9 = np.ascontiguousarray(tris, np.float32)
        r = np.ascontiguousarray(rays)
        count = len(r)
        ids, t, again = np.zeros(count, np.int32), np.zeros(count, np.float32), np.zeros(1, np.int32)
        error = self.lib.wide_trace(self.n, _p(self.nodes), _p(self.wide), _p(self.wide_leaf), _p(t9), len(t9),
                                    _p(r), count, int(any_hit), group, _p(ids), _p(t), _p(again))
        return ids, t, int(again[0]), error


def check(model, boxes, ids, tris, rays, groups=(1, 4, 16)):
    tree = oracle.OracleBvh(boxes, ids)
    m = model(tree)
    assert m.fill_error == 0
    want = tree.trace_closest(tris, rays)
    for g in groups:
        got, t, again, error = m.trace(tris, rays, group=g)
        assert error == 0
        assert np.array_equal(got, want["ids"]), g
        hit = want["ids"] >= 0
        assert np.array_equal(t[hit].view(np.uint32), want["t"][hit].view(np.uint32)), g
        assert again <= len(rays) // 4  # flat boxes: entries a rounding above their hits
        occ, _, _, error = m.trace(tris, rays, any_hit=True, group=g)
        assert error == 0 and np.array_equal(occ >= 0, hit), g


@pytest.mark.parametrize("case", ["soup2000", "clustered1500", "identical64", "flat300", "sparse_ids777", "tiny2", "tiny3",
                                  "tiny7", "rounding4", "signed_zero4000"])
def test_golden_trees(model, case):
    g = load_golden(f"lbvh_{case}")
    check(model, g["boxes"], g["ids"], g["tri_by_id"], g["rays"])


def test_random_soup_and_axis_parallel_rays(model):
    tris = W.soup(1 << 12, seed=0x4C5558)
    rays = W.rays(2048, seed=0x4C555A)
    r = rays.view(np.float32).reshape(len(rays), -1)
    r[::5, 3] = 0  # one, then two parallel axes
    r[::10, 4] = 0
    check(model, W.triangle_boxes(tris), None, tris, rays)


def meets(box, ray, t_max):
    """The reference's slab test, in its own float operations."""
    o, d = ray[0:3], ray[3:6]
    near, far = np.float32(ray[6]), np.float32(t_max)
    for a in range(3):
        inv = np.float32(1) / d[a]
        lo, hi = (box[3 + a], box[a]) if inv < 0 else (box[a], box[3 + a])
        near, far = max(near, (lo - o[a]) * inv), min(far, (hi - o[a]) * inv)
    return not near > far


@pytest.mark.parametrize("bad_id", [2000, 0x7FFFFFFF])
def test_leaf_ids_out_of_range_are_reported_where_the_leaf_box_is_met(model, bad_id):
    """An id at or above the triangle count is an error for exactly the rays that
    meet its leaf's own box no farther than their hit (any hit: that find none), not
    for those that only meet the wider byte box."""
    g = load_golden("lbvh_soup2000")
    tris = g["tri_by_id"]
    boxes, ids = g["boxes"].copy(), g["ids"].astype(np.int32).copy()
    k = int(np.argmax(np.prod(boxes[:, 3:] - boxes[:, :3], axis=1)))
    boxes[k] = [0.3, 0.3, 0.3, 0.7, 0.7, 0.7]  # a large leaf that many rays meet
    rest = tris.copy()
    rest[ids[k]] = 0  # what the oracle walks: never hit there
    want = oracle.OracleBvh(boxes, ids).trace_closest(rest, g["rays"][:400])
    ids[k] = bad_id
    m = model(oracle.OracleBvh(boxes, ids))
    seen = {True: 0, False: 0}
    for i in range(400):
        ray = g["rays"][i : i + 1]
        hit = want["ids"][i] >= 0
        met = meets(boxes[k], ray[0], want["t"][i] if hit else ray[0][7])
        for group in (1, 16):
            got, t, _, error = m.trace(tris, ray, group=group)
            assert error == (PRIM_RANGE if met else 0), (i, group)
            assert got[0] == want["ids"][i]
            occ, _, _, error = m.trace(tris, ray, any_hit=True, group=group)
            assert (occ[0] >= 0) == hit and error == (PRIM_RANGE if met and not hit else 0), (i, group)
        seen[met] += 1
    assert min(seen.values()) > 10


def damaged(kind):
    """Run in a process of its own: prints the error bits."""
    g = load_golden("lbvh_soup2000")
    tris, rays = g["tri_by_id"], g["rays"][:256]
    tree = oracle.OracleBvh(g["boxes"], g["ids"])
    assert (tree.trace_closest(tris, rays)["ids"] >= 0).sum() > 50

    def links(m):  # children out of range: their records must hold no stale position
        m.left[7] = 0x20000000
        m.right[150] = 0x80000000 | 0x20000000

    def places(m):
        m.pre_leaf[::3] = -5
        m.pre_leaf[1::3] = 0x40000000

    m = WideModel(tree, {"links": links, "places": places}.get(kind))
    if kind == "leaf positions":
        m.wide_leaf[:] = 0x40000000
    if kind == "negative positions":
        m.wide_leaf[:] = -0x40000000
    error = m.fill_error
    for group in (1, 8):
        error |= m.trace(tris, rays, group=group)[3] | m.trace(tris, rays, any_hit=True, group=group)[3]
    print("error", error, flush=True)


@pytest.mark.parametrize("kind", ["links", "places", "leaf positions", "negative positions"])
def test_damaged_arrays_end_in_an_error_bit(model, kind):
    r = subprocess.run([sys.executable, __file__, kind], capture_output=True, text=True, timeout=120,
                       env={**os.environ, "PYTHONPATH": str(ROOT)})
    assert r.returncode == 0, (r.returncode, r.stderr)
    assert r.stdout.split() == ["error", str(WALK_ORDER)]


if __name__ == "__main__":
    damaged(sys.argv[1])
