"""GPU: traversal copies made for their first reader (records for rays, pairs for
overlaps) against fresh trees, over refits, two streams and captured graphs."""

import ctypes

import numpy as np
import pytest

from lux_amd import workloads as W

pytestmark = pytest.mark.gpu

N, M, MAX_PAIRS = 20011, 3001, 1 << 18


class Tree:
    """A handle with its buffers, and the answers of a fresh tree over the same triangles."""

    def __init__(self, lb, seed):
        from lux_amd import abi

        self.lb, self.abi = lb, abi
        self.tris = W.soup(N, seed=seed, edge=(0.01, 0.05))
        self.d_tris = lb.DeviceArray.from_numpy(self.tris)
        self.rays = lb.DeviceArray.from_numpy(W.rays(M, seed=seed + 1))
        self.hits = lb.DeviceArray.from_numpy(np.zeros(2 * M, np.int32))
        self.pairs, self.found = lb.DeviceArray(8 * MAX_PAIRS), lb.DeviceArray(4)
        self.bvh = lb.GpuBvh()

    def move(self, seed):
        self.tris = W.jitter(self.tris, sigma=5e-3, seed=seed)
        self.abi.call("lux_hip_memcpy_htod", self.d_tris.ptr, self.abi.ptr(self.tris),
                      ctypes.c_size_t(self.tris.nbytes))

    def trace(self, stream=None):
        self.abi.call("lux_hip_trace_closest_device", self.bvh.handle, self.d_tris.ptr, N, self.rays.ptr, M,
                      self.hits.ptr, stream)

    def overlap(self, stream=None):
        self.abi.call("lux_hip_overlap_self_device", self.bvh.handle, MAX_PAIRS, self.pairs.ptr, self.found.ptr, stream)

    def build(self, stream=None):
        self.bvh.build_triangles_device(self.d_tris, N, stream=stream)

    def refit(self, stream=None):
        self.bvh.refit_triangles_device(self.d_tris, N, stream=stream)

    def check(self, rays=True, pairs=True):
        """Against a tree of its own, built from the first triangles' topology or not:
        closest hits and pair sets do not depend on the tree."""
        self.lb.synchronize()
        fresh = self.lb.GpuBvh()
        fresh.build_triangles_device(self.d_tris, N)
        own = self.bvh
        if rays:
            got = self.hits.to_numpy(np.int32, 2 * M)
            self.bvh = fresh
            self.trace()
            self.bvh = own
            assert (got[0::2] >= 0).sum() > 100
            assert np.array_equal(got, self.hits.to_numpy(np.int32, 2 * M))
        if pairs:
            k = int(self.found.to_numpy(np.int32, 1)[0])
            got = self.pairs.to_numpy(np.int32, (MAX_PAIRS, 2))[:k]
            self.bvh = fresh
            self.overlap()
            self.bvh = own
            assert 1000 < k <= MAX_PAIRS and k == int(self.found.to_numpy(np.int32, 1)[0])
            want = self.pairs.to_numpy(np.int32, (MAX_PAIRS, 2))[:k]
            assert np.array_equal(got[np.lexsort(got.T)], want[np.lexsort(want.T)])
        fresh.close()


class Hip:
    """The few runtime calls a program that captures graphs makes."""

    def __init__(self):
        self.lib = ctypes.CDLL("libamdhip64.so.7")

    def __call__(self, name, *args):
        assert getattr(self.lib, name)(*args) == 0, name

    def stream(self):
        s = ctypes.c_void_p()
        self("hipStreamCreateWithFlags", ctypes.byref(s), 1)  # non-blocking
        return s

    def capture(self, stream, fn):
        g, e = ctypes.c_void_p(), ctypes.c_void_p()
        self("hipStreamBeginCapture", stream, 1)  # thread-local
        fn()
        self("hipStreamEndCapture", stream, ctypes.byref(g))
        self("hipGraphInstantiate", ctypes.byref(e), g, None, None, ctypes.c_size_t(0))
        return e

    def replay(self, graph, stream):
        self("hipGraphLaunch", graph, stream)
        self("hipStreamSynchronize", stream)


def test_queries_and_refits_in_any_order(gpu):
    print("case: copies, order", flush=True)
    t = Tree(gpu, 21)
    t.build()
    t.overlap()
    t.trace()
    t.check()
    for k, order in enumerate(["trace", "overlap", "trace overlap", "overlap trace", "overlap trace overlap"]):
        t.move(31 + k)
        t.refit()
        for op in order.split():
            getattr(t, op)()
        t.check(rays="trace" in order, pairs="overlap" in order)


def test_two_streams_on_one_handle(gpu):
    """Each call on the other stream: what one makes the next one reads."""
    print("case: copies, two streams", flush=True)
    hip = Hip()
    a, b = hip.stream(), hip.stream()
    t = Tree(gpu, 22)
    t.build(a)
    for k in range(4):
        t.trace(b)
        t.overlap(a)
        t.check()
        t.move(41 + k)
        t.refit(b if k % 2 else a)


def test_captured_trace_replayed_after_refits(gpu):
    """A graph that holds only the query reads the records of the tree as it is when
    it is replayed."""
    print("case: copies, captured trace", flush=True)
    hip = Hip()
    s = hip.stream()
    t = Tree(gpu, 23)
    t.build(s)
    t.trace(s)
    t.check(pairs=False)
    graph = hip.capture(s, lambda: t.trace(s))
    for k in range(4):
        t.move(51 + k)
        t.refit(s)
        hip.replay(graph, s)
        t.check(pairs=False)
        t.overlap(s)
        t.check(rays=False)


def test_captured_refit_with_queries_outside(gpu):
    """A graph that holds only the refit, and one with its query: queries after each
    replay read the moved tree."""
    print("case: copies, captured refit", flush=True)
    hip = Hip()
    s = hip.stream()
    t = Tree(gpu, 24)
    t.build(s)
    t.trace(s)
    t.overlap(s)
    t.check()
    refit = hip.capture(s, lambda: t.refit(s))
    both = hip.capture(s, lambda: (t.refit(s), t.trace(s)))
    for k in range(3):
        t.move(61 + k)
        hip.replay(refit, s)
        t.trace(s)
        t.overlap(s)
        t.check()
        t.move(71 + k)
        hip.replay(both, s)
        t.check(pairs=False)
        t.overlap(s)
        t.check(rays=False)
