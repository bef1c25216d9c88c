"""Scenes of test_host_runtime.py: the library's host code stepped on the CPU over
tests/hip_stub.cpp. Each scene runs in a process of its own (the stub's symbols
must be there before the library is loaded):

    python tests/host_runtime.py SCENE

prints one JSON line. Kernels do not run; `Stub` sees every launch and does in
host memory what a scene depends on (clears).
"""

import ctypes
import json
import sys
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))

STUB = Path(__file__).resolve().parent / "_build" / "libhip_stub.so"
CALLBACK = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p))


class Stub:
    def __init__(self):
        self.lib = ctypes.CDLL(str(STUB), mode=ctypes.RTLD_GLOBAL)
        self.lib.stub_live_bytes.restype = ctypes.c_uint64
        self.launches = []
        self.hooks = []  # (part of a kernel's name, function(stub, args))
        self._cb = CALLBACK(self._launch)
        self.lib.stub_on_launch(self._cb)

    def _launch(self, name, stream, args):
        name = name.decode()
        self.launches.append(name)
        self.stream = stream or 0
        if "k_zero_u32" in name:  # (uint32_t* p, int n)
            ctypes.memset(ptr(args, 0), 0, 4 * i32(args, 1))
        if "k_clear_tree" in name:  # (status, words, tickets, counter, info)
            ctypes.memset(ptr(args, 0), 0, 8 * i32(args, 1))
            for k, size in ((2, 16), (3, 16), (4, 64)):
                ctypes.memset(ptr(args, k), 0, size)
        if "k_clear_counts" in name:  # (counts, rays)
            ctypes.memset(ptr(args, 0), 0, 16)
            ctypes.memset(ptr(args, 1), 0, 16)
        for part, fn in self.hooks:
            if part in name:
                fn(args)


def ptr(args, k):
    return ctypes.cast(args[k], ctypes.POINTER(ctypes.c_void_p))[0]


def i32(args, k):
    return ctypes.cast(args[k], ctypes.POINTER(ctypes.c_int32))[0]


def words(address, count, dtype=np.uint32):
    n = count * np.dtype(dtype).itemsize
    return np.frombuffer((ctypes.c_uint8 * n).from_address(address), dtype)


class SortWatch:
    """Every radix pass must find its tile ticket at zero and, on a tree's first
    pass, no look-back word of an earlier owner of the memory."""

    def __init__(self, stub):
        self.bad, self.passes = [], 0
        stub.hooks.append(("k_sort_pass", self.see))

    def see(self, args):
        self.passes += 1
        status, ticket, epoch, tiles = ptr(args, 7), ptr(args, 8), i32(args, 9), i32(args, 10)
        if words(ticket, 1)[0] != 0:
            self.bad.append(f"ticket {words(ticket, 1)[0]}")
        if epoch == 1 and words(status, tiles * 256, np.uint64).any():
            self.bad.append("look-back words of another sort")


def sphere(k, freq=6):
    from lux_amd import scenes

    return scenes.displaced_icosphere(freq=freq + k, seed=0x4C5700 + k, width=16, height=16)


def small_engine():
    from lux_amd import render

    render.set_tuning(capacity=4096, grid=8, block=256, use_graph=0)
    return render


def job(i):
    return dict(width=16, height=16, spp=2, depth=2, seed=i)


def tight_stream(render, scs, order, verts):
    """The scenes served under a budget that holds two and a half of them."""
    sizes = [sc.info()[2] for sc in scs]
    probe = render.Server(hbm_budget=1 << 40, slice_spp=8)
    probe.run([scs[0]], [job(0)], [0.0], want_films=False)
    fixed = probe.stats()["peak_bytes"] - sizes[0]
    probe.close()
    sv = render.Server(hbm_budget=fixed + int(2.5 * max(sizes)), slice_spp=8)
    sv.run([scs[k] for k in order], [job(i) for i in range(len(order))], [0.001 * i for i in range(len(order))],
           vertices=verts, want_films=False)
    st = sv.stats()
    sv.close()
    return st


def clears(stub):
    """Builds (handles, scenes, a served stream with evictions and restores) over
    memory that holds old bytes."""
    from lux_amd import abi, lbvh, workloads as W

    watch = SortWatch(stub)
    tris = W.soup(3000, seed=1)
    bvh = lbvh.GpuBvh()
    boxes = lbvh.DeviceArray.from_numpy(W.triangle_boxes(tris))
    ids = lbvh.DeviceArray.from_numpy(np.arange(3000, dtype=np.int32))
    bvh.build_device(boxes, ids, 3000)
    rays = lbvh.DeviceArray(32 * ((1 << 21) + 3))
    hits = lbvh.DeviceArray(8 * ((1 << 21) + 3))
    d_tris = lbvh.DeviceArray.from_numpy(tris)
    abi.call("lux_hip_trace_closest_device", bvh.handle, d_tris.ptr, 3000, rays.ptr, (1 << 21) + 3, hits.ptr,
             None)  # sorted: the ray-order scratch
    render = small_engine()
    dicts = [sphere(k) for k in range(5)]
    scs = [render.Scene(d, deferred=True) for d in dicts]
    order = [0, 1, 2, 3, 4, 0, 2, 4, 1, 3, 0]
    verts = [None] * len(order)
    verts[5], verts[8] = dicts[0]["vertices"] + np.float32(1e-3), dicts[1]["vertices"] + np.float32(1e-3)
    st = tight_stream(render, scs, order, verts)
    return {"bad": watch.bad, "passes": watch.passes, "null_writes": stub.lib.stub_null_writes(),
            "evictions": st["evictions"], "uploads": st["uploads"], "completed": st["completed"]}


class ErrorBits:
    """Sets a device error bit of one tree as a launch's effect."""

    def __init__(self, stub):
        self.infos, self.build, self.render = [], None, None
        stub.hooks.append(("k_copies", self.built))
        stub.hooks.append(("k_flush", self.flushed))

    def built(self, args):
        info = ptr(args, 12)
        self.infos.append(info)
        if self.build == len(self.infos):
            words(info + 32, 1)[0] = 2

    def flushed(self, args):
        if self.render is not None:
            words(self.infos[self.render] + 32, 1)[0] = 2
            self.render = None


def status_of(fn):
    from lux_amd.abi import LuxError

    try:
        fn()
    except LuxError as e:
        return e.status
    return 0


def errors(stub):
    """Failed device checks of a build or a render reach the caller, and the server
    goes on."""
    from lux_amd import lbvh

    bits = ErrorBits(stub)
    render = small_engine()
    out = {}
    bits.build = 1
    out["create"] = status_of(lambda: render.Scene(sphere(0)))
    a = render.Scene(sphere(0))
    bits.build = len(bits.infos) + 1
    out["update"] = status_of(lambda: a.update_vertices(sphere(0)["vertices"]))
    out["update_again"] = status_of(lambda: a.update_vertices(sphere(0)["vertices"]))
    base = stub.lib.stub_live_bytes()
    cold = render.Scene(sphere(1), deferred=True)
    bits.build = len(bits.infos) + 1
    out["first_use"] = status_of(lambda: cold.render(16, 16, 1, 1))
    out["kept"] = stub.lib.stub_live_bytes() - base  # nothing of the failed build
    sv = render.Server(slice_spp=8)

    def run(scs):
        return sv.run(scs, [job(i) for i in range(len(scs))], [0.0] * len(scs), want_films=False)

    bits.build = len(bits.infos) + 1
    out["served_upload"] = status_of(lambda: run([a, cold, a]))
    out["served_again"] = status_of(lambda: run([a, cold, a]))
    bits.render = bits.infos.index(bits.infos[-1])  # the scene just uploaded
    out["served_render"] = status_of(lambda: run([a, cold, a]))
    out["served_after"] = status_of(lambda: run([a, cold, a]))
    # by polling: every request is reported, the failed one's result is the error
    other = render.Scene(sphere(2), deferred=True)
    bits.build = len(bits.infos) + 1
    ids = [sv.submit(a, job(1)), sv.submit(other, job(2))]
    done = []
    for _ in range(100000):
        done += sv.poll(block=True)
        if len(done) == 2:
            break
    out["polled"] = [status_of(lambda i=i: sv.result(i)) for i in ids]
    st = sv.stats()
    out["open"] = st["submitted"] - st["completed"]
    out["destroy"] = status_of(lambda: render.call("lux_hip_scene_destroy", other.handle))
    other.handle = None
    return out


def bytes_held(stub):
    """Device memory a scene reports (resident, and deferred before it is built)
    against what it allocates."""
    render = small_engine()
    dicts = [sphere(k, freq) for k, freq in ((0, 2), (1, 8), (2, 24))]
    lit = dict(dicts[1])
    lit["lights"] = [{"kind": "image_infinite", "color": (1, 1, 1), "image": np.ones((16, 32, 3), np.float32)},
                     {"kind": "point", "vector": (0, 2, 0), "color": (1, 1, 1)}]
    out = []
    for d in dicts + [lit]:
        before = stub.lib.stub_live_bytes()
        sc = render.Scene(d)
        deferred = render.Scene(d, deferred=True)
        out.append([sc.info()[2], deferred.info()[2], stub.lib.stub_live_bytes() - before, len(d["indices"])])
        deferred.close()
        sc.close()
        assert stub.lib.stub_live_bytes() == before
    return {"scenes": out}


def lost_instances(stub):
    """set_instances with more instances in view than before (two of three had empty
    bounds) that runs out of memory at each of its allocations in turn: queries are
    refused until it has succeeded."""
    from lux_amd import lbvh, two_level, workloads as W

    lbvh.init()
    tris = W.soup(40, seed=3).reshape(-1, 9)
    mesh = np.array([0, 1, 0], np.int32)
    m = np.stack([W.affine(None, (1, 1, 1), (0.5 * k, 0, 0)) for k in range(3)]).astype(np.float32)
    offsets = np.array([0, 25, 40], np.int32)
    inst = two_level.make_instances(mesh, m, tris, offsets)
    first = inst.copy()
    first["world_bounds"][1:] = [1, 1, 1, -1, -1, -1]
    sc = two_level.TwoLevelScene(tris, offsets, first)
    rays = W.rays(10, seed=4)
    out = []
    for k in range(60):
        stub.lib.stub_fail_alloc_after(k)
        failed = status_of(lambda: sc.set_instances(inst))
        stub.lib.stub_fail_alloc_after(-1)
        out.append([failed, status_of(lambda: sc.intersect(rays))])
        if not failed:
            break
    return {"tries": out}


def copies(stub):
    """Which traversal copies each call makes (r: records, p: pairs)."""
    from lux_amd import abi, lbvh, workloads as W

    made = []

    def see(args):
        wide = i32(args, 1)
        made.append(("r" if wide else "") + ("p" if stub.lib.stub_grid() > wide else ""))

    stub.hooks.append(("k_copies", see))
    n = 5000
    tris = W.soup(n, seed=1)
    d_tris, rays = lbvh.DeviceArray.from_numpy(tris), lbvh.DeviceArray(36 * 64)
    out = lbvh.DeviceArray(8 * 4096)
    bvh = lbvh.GpuBvh()
    calls = {
        "build": lambda: bvh.build_triangles_device(d_tris, n),
        "refit": lambda: bvh.refit_triangles_device(d_tris, n),
        "trace": lambda: abi.call("lux_hip_trace_closest_device", bvh.handle, d_tris.ptr, n, rays.ptr, 64, out.ptr,
                                  None),
        "any": lambda: abi.call("lux_hip_trace_any_device", bvh.handle, d_tris.ptr, n, rays.ptr, 64, out.ptr, None),
        "overlap": lambda: abi.call("lux_hip_overlap_self_device", bvh.handle, 64, out.ptr, rays.ptr, None),
    }

    def run(text):
        got = []
        for word in text.split():
            made.clear()
            stub.lib.stub_capturing(int(word.startswith("graph:")))
            calls[word.split(":")[-1]]()
            stub.lib.stub_capturing(0)
            got.append("+".join(made) or "-")
        return got

    first = run("build trace any trace overlap overlap refit refit any overlap trace build overlap")
    recorded = run("graph:refit trace overlap trace refit graph:trace trace refit trace overlap graph:build graph:trace")
    d = sphere(0)
    made.clear()
    render = small_engine()
    sc = render.Scene(d)
    sc.update_vertices(d["vertices"])
    return {"first": first, "recorded": recorded, "scene": list(made)}


def query_launches(stub):
    """The kernel and its threads for 1000 rays over trees of few triangles."""
    from lux_amd import abi, lbvh, workloads as W

    rays, hits = lbvh.DeviceArray(36 * 1000), lbvh.DeviceArray(8 * 1000)
    seen = []
    stub.hooks.append(("7k_trace", lambda args: seen.append(["k_trace", stub.lib.stub_grid() * stub.lib.stub_block()])))
    stub.hooks.append(("13k_trace_parts", lambda args: seen.append(["parts", stub.lib.stub_grid() * stub.lib.stub_block()])))
    stub.hooks.append(("16k_trace_preorder", lambda args: seen.append(["preorder", 0])))
    out = {}
    for n in (1, 2, 16, 17, 300):
        d = lbvh.DeviceArray.from_numpy(W.soup(n, seed=1))
        bvh = lbvh.GpuBvh()
        bvh.build_triangles_device(d, n)
        seen.clear()
        abi.call("lux_hip_trace_closest_device", bvh.handle, d.ptr, n, rays.ptr, 1000, hits.ptr, None)
        out[n] = seen[-1]
    return out


def trace_launches(stub):
    """k_trace's walk and threads, as [walk, threads] of the first launch of each
    render."""
    from lux_amd import scenes

    render = small_engine()
    seen = []
    stub.hooks.append(("7k_traceILi", lambda args: seen.append([stub.launches[-1].split("ELi")[1][0],
                                                                stub.lib.stub_grid() * stub.lib.stub_block()])))
    out = {}
    made = {"room": scenes.instanced_room(64, 48), "box": scenes.cornell(64, 48),
            "sphere": scenes.displaced_icosphere(freq=8, seed=1, width=64, height=48)}
    for name, d in made.items():
        sc = render.Scene(d)
        for mode, text in ((render.PLAIN, "plain"), (render.WAVEFRONT, "wave")):
            for preorder in (False, True):
                render.set_tuning(preorder_walk=preorder)
                seen.clear()
                sc.render(64, 48, 1, 1, mode=mode)
                out[f"{name} {text}{' preorder' if preorder else ''}"] = seen[0]
    return out


def failed_builds(stub):
    """A build that runs out of memory at each of its allocations in turn, then the
    same build again with memory to spare and queries over it: the arrays its kernels
    are given."""
    from lux_amd import abi, lbvh, workloads as W

    n = 300
    d_tris, rays, out = lbvh.DeviceArray.from_numpy(W.soup(n, seed=1)), lbvh.DeviceArray(36), lbvh.DeviceArray(8)
    null = []
    want = {"k_copies": range(2, 9), "11k_sort_pass": (0, 1, 2, 3, 6, 7, 8, 11), "7k_local": (1, 2, 6, 7, 8, 9, 10)}
    for name, ks in want.items():
        stub.hooks.append((name, lambda args, name=name, ks=ks: null.extend([name, k] for k in ks if not ptr(args, k))))
    base = stub.lib.stub_live_bytes()
    tries, left = [], []
    for k in range(60):
        bvh = lbvh.GpuBvh()
        stub.lib.stub_fail_alloc_after(k)
        tries.append(status_of(lambda: bvh.build_triangles_device(d_tris, n)))
        stub.lib.stub_fail_alloc_after(-1)
        left.append(stub.lib.stub_live_bytes() - base if tries[-1] else 0)
        null.clear()
        bvh.build_triangles_device(d_tris, n - 1)
        abi.call("lux_hip_trace_closest_device", bvh.handle, d_tris.ptr, n, rays.ptr, 1, out.ptr, None)
        assert null == [], (k, null)
        bvh.close()
        if not tries[-1]:
            break
    # the scratch of the ray order, and a renderer's path buffer
    m = (1 << 21) + 1
    bvh, rays, out = lbvh.GpuBvh(), lbvh.DeviceArray(36 * m), lbvh.DeviceArray(8 * m)
    bvh.build_triangles_device(d_tris, n)
    render = small_engine()
    sc = render.Scene(sphere(0))
    film = lbvh.DeviceArray(12 * 256)
    rs = render.settings(width=16, height=16, spp=1, depth=1)
    stub.hooks.append(("k_generate", lambda args: null.extend(["k_generate", k] for k in range(3) if not ptr(args, k))))
    later = {
        "order": lambda: abi.call("lux_hip_trace_closest_device", bvh.handle, d_tris.ptr, n, rays.ptr, m, out.ptr,
                                  None),
        "paths": lambda: abi.call("lux_hip_render_device", sc.handle, ctypes.byref(rs), film.ptr, None),
    }
    counts = {}
    for name, call in later.items():
        base = stub.lib.stub_live_bytes()
        for k in range(20):
            stub.lib.stub_fail_alloc_after(k)
            failed = status_of(call)
            stub.lib.stub_fail_alloc_after(-1)
            if not failed:
                break
            left.append(stub.lib.stub_live_bytes() - base)
        counts[name] = k
        null.clear()
        call()
        assert null == [], (name, null)
    return {"tries": tries, "left": left, "later": counts}


def two_threads(stub):
    """Two threads that query one tree on streams of their own right after a refit:
    every walk must be ordered behind the launch that made its records."""
    import threading

    from lux_amd import abi, lbvh, workloads as W

    for fn in (stub.lib.stub_launches, stub.lib.stub_waited):
        fn.restype, fn.argtypes = ctypes.c_long, [ctypes.c_void_p]
    n = 300
    d_tris, rays, out = lbvh.DeviceArray.from_numpy(W.soup(n, seed=1)), lbvh.DeviceArray(36), lbvh.DeviceArray(8)
    bvh = lbvh.GpuBvh()
    bvh.build_triangles_device(d_tris, n)
    streams = [ctypes.c_void_p(0xA000), ctypes.c_void_p(0xB000)]
    here = threading.local()
    made, late, walks = {}, [], [0]

    def see(name, stream):  # in the launching thread
        if "k_copies" in name:
            made[0] = (stream, stub.lib.stub_launches(stream))
        elif "13k_trace_parts" in name:
            walks[0] += 1
            s, index = made[0]
            if s != stream and stub.lib.stub_waited(s) < index:
                late.append(walks[0])

    cb = CALLBACK(lambda name, stream, args: see(name.decode(), stream or 0))
    stub.lib.stub_on_launch(cb)
    start, stop = threading.Barrier(2), threading.Barrier(2)

    def work(k):
        for _ in range(400):
            if k == 0:
                bvh.refit_triangles_device(d_tris, n, stream=streams[0])
            start.wait()
            abi.call("lux_hip_trace_closest_device", bvh.handle, d_tris.ptr, n, rays.ptr, 1, out.ptr, streams[k])
            stop.wait()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    return {"walks": walks[0], "late": len(late)}


def host_queries(stub):
    """Queries from and to host arrays, with another thread's call on a stream of its
    own between their walk and the copy of their results: launches and copies of their
    own stream that they did not wait for."""
    import threading

    from lux_amd import abi, lbvh, workloads as W

    for fn in (stub.lib.stub_launches, stub.lib.stub_waited):
        fn.restype, fn.argtypes = ctypes.c_long, [ctypes.c_void_p]
    n = 300
    soup, host_rays = W.soup(n, seed=1), W.rays(10, seed=4)
    d_tris, rays, out = lbvh.DeviceArray.from_numpy(soup), lbvh.DeviceArray(36), lbvh.DeviceArray(8)
    bvh = lbvh.GpuBvh()
    bvh.build_triangles_device(d_tris, n)
    own = stub.stream
    calls = [0]

    def other(stream):
        calls[0] += 1
        t = threading.Thread(target=abi.call, args=("lux_hip_trace_closest_device", bvh.handle, d_tris.ptr, n, rays.ptr, 1,
                                                    out.ptr, ctypes.c_void_p(0xA000)))
        t.start()
        t.join()

    cb = ctypes.CFUNCTYPE(None, ctypes.c_void_p)(other)
    stub.lib.stub_on_download(cb)
    open_work = []
    for query in (lbvh.intersect_gpu_bvh_stackless, lbvh.trace_any):
        query(bvh, soup, host_rays)
        open_work.append(stub.lib.stub_launches(own) - stub.lib.stub_waited(own))
    stub.lib.stub_on_download(None)
    return {"calls": calls[0], "open": open_work}


if __name__ == "__main__":
    print(json.dumps(globals()[sys.argv[1]](Stub())))
