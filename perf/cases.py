"""Workloads of this framework through its public entry points, for timing and
for comparing outputs.

The listed cases are what programs call it for: ray queries against one tree
(closest hit, any hit), trees rebuilt or refitted every frame, box contacts,
instanced scenes, path-traced images (a preview, a full frame, a batch of many
scenes) and the encoding of a finished film. Sizes are those of the
repository's own benchmark and tests or lie between them, odd ones included.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs and handles a program holds before the call
    run(state)          one pass, returning its outputs
    work(case)          bytes and operations the pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the outputs in 64 bits by plain torch, where possible

Buffers are torch tensors handed over by address; the library's own stream is
used unless torch works on the outputs too (contacts).
"""

import ctypes
import math

import numpy as np
import torch

from lux_amd import abi, film, lbvh, render, scenes, two_level, workloads

DEVICE = "cuda"


# ---- the cases -------------------------------------------------------------------
def listed():
    return [
        # the smallest program: a mesh of a few hundred triangles, one thousand
        # picking rays (an editor, a unit of a game level): latency and launches
        {"name": "pick_small", "kind": "build", "tris": 777, "rays": 1000},
        # a new tree every frame for a large deforming mesh, probed by a few rays
        {"name": "rebuild_large", "kind": "build", "tris": 1 << 20, "rays": 1 << 14},
        # a mesh whose vertices move: boxes refitted, then queried (odd sizes)
        {"name": "refit_frame", "kind": "refit", "tris": 262147, "rays": 65537},
        # primary rays of a camera: coherent directions and origins
        {"name": "query_camera", "kind": "query", "op": "closest", "shape": "sphere", "tris": 81920, "rays": 1280 * 720},
        # incoherent closest hits (the LBVH microbenchmark)
        {"name": "query_random", "kind": "query", "op": "closest", "shape": "soup", "tris": 1 << 20, "rays": 1 << 22},
        # visibility of point pairs: any hit with finite segments
        {"name": "visibility", "kind": "query", "op": "any", "shape": "soup", "tris": 500009, "rays": 1500007},
        # broad phase: a tree over moving boxes each step, its overlaps with a static one
        {"name": "contacts", "kind": "contacts", "op": "cross", "tris": 1 << 20, "boxes": 100000},
        # rays through an instanced scene (two levels)
        {"name": "instances", "kind": "two_level", "op": "closest", "meshes": 4, "tris": 1 << 16, "instances": 64,
         "rays": 1 << 20},
        # an interactive preview: few paths, latency of the bounce loop
        {"name": "preview", "kind": "render", "scene": "cornell", "width": 128, "height": 96, "spp": 4, "depth": 4},
        # a frame of one detailed scene with glass, glossy and diffuse materials
        {"name": "frame", "kind": "render", "scene": "sphere", "freq": 128, "width": 1024, "height": 1024, "spp": 16,
         "depth": 8},
        # several users' images in one call: four meshes of different size and an instanced scene
        {"name": "batch", "kind": "batch", "meshes": 4, "freq": 96, "side": 512, "spp": 8, "depth": 6},
        # the finished film as bytes, 4K
        {"name": "film_bytes", "kind": "film", "format": "ppm", "width": 3840, "height": 2160, "spp": 64},
    ]


def _log(rng, lo, hi):
    """A whole number, uniform over its logarithm, odd about half of the time."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n | 1 if rng.random() < 0.5 else n))


def draw(rng):
    kind = rng.choice(["build", "refit", "query", "query", "contacts", "two_level", "render", "render", "batch",
                       "film"])
    if kind == "build":
        return {"kind": kind, "tris": _log(rng, 200, 1 << 20), "rays": _log(rng, 500, 1 << 15)}
    if kind == "refit":
        return {"kind": kind, "tris": _log(rng, 500, 1 << 20), "rays": _log(rng, 500, 1 << 17)}
    if kind == "query":
        op, shape = rng.choice(["closest", "any"]), rng.choice(["soup", "sphere"])
        tris = _log(rng, 300, 1 << 20) if shape == "soup" else 20 * _log(rng, 8, 160) ** 2
        return {"kind": kind, "op": op, "shape": shape, "tris": tris, "rays": _log(rng, 500, 1 << 21)}
    if kind == "contacts":
        return {"kind": kind, "op": rng.choice(["cross", "self"]), "tris": _log(rng, 2000, 1 << 20),
                "boxes": _log(rng, 1000, 200000)}
    if kind == "two_level":
        return {"kind": kind, "op": rng.choice(["closest", "any"]), "meshes": rng.randint(1, 6),
                "tris": _log(rng, 200, 1 << 16), "instances": _log(rng, 2, 100), "rays": _log(rng, 1000, 1 << 20)}
    if kind == "render":
        scene = rng.choice(["cornell", "sphere", "instanced"])
        c = {"kind": kind, "scene": scene, "width": _log(rng, 48, 640), "height": _log(rng, 48, 640),
             "spp": _log(rng, 1, 16), "depth": rng.randint(2, 8)}
        if scene != "cornell":
            c["freq"] = _log(rng, 8, 100 if scene == "sphere" else 40)
        return c
    if kind == "batch":
        return {"kind": kind, "meshes": rng.randint(2, 5), "freq": _log(rng, 10, 90), "side": _log(rng, 64, 400),
                "spp": _log(rng, 2, 8), "depth": rng.randint(3, 8)}
    return {"kind": kind, "format": rng.choice(["ppm", "pfm"]), "width": _log(rng, 100, 3840),
            "height": _log(rng, 100, 2160), "spp": _log(rng, 1, 256)}


# ---- inputs ----------------------------------------------------------------------
class Buffer:
    """A torch tensor as the library takes device arrays: by its address."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _generator(seed, part):
    return torch.Generator(device=DEVICE).manual_seed(int(seed) * 16 + part)


def _directions(n, g):
    d = torch.randn(n, 3, generator=g, device=DEVICE, dtype=torch.float64)
    return d / d.norm(dim=1, keepdim=True)


def _soup(n, seed, part=0, per=None):
    """n triangles in the unit cube, edges 0.1 to 1 of the mean spacing of
    `per` (n) points, the density of the LBVH microbenchmark: (n, 9)."""
    g = _generator(seed, part)
    spacing = float(per or n) ** (-1.0 / 3.0)
    v0 = torch.rand(n, 3, generator=g, device=DEVICE, dtype=torch.float64)
    edge = (0.1 + 0.9 * torch.rand(n, 2, generator=g, device=DEVICE, dtype=torch.float64)) * spacing
    v1 = v0 + edge[:, :1] * _directions(n, g)
    v2 = v0 + edge[:, 1:] * _directions(n, g)
    return torch.cat([v0, v1, v2], 1).float().contiguous()


def _boxes(tris):
    t = tris.view(-1, 3, 3)
    return torch.cat([t.amin(1), t.amax(1)], 1).contiguous()


def _moved(tris, seed):
    """The soup with every vertex moved by a tenth of the mean spacing."""
    g = _generator(seed, 9)
    step = 0.1 * float(len(tris)) ** (-1.0 / 3.0)
    return (tris + step * torch.randn(tris.shape, generator=g, device=DEVICE)).contiguous()


def _ray_array(o, d, t_max):
    r = torch.zeros(len(o), 9, device=DEVICE)
    r[:, 0:3] = o
    r[:, 3:6] = d
    r[:, 7] = t_max
    return r


def _random_rays(n, seed, segments=False):
    """Origins in the unit cube, directions on the sphere; segments end 0.05 to
    0.5 away."""
    g = _generator(seed, 1)
    o = torch.rand(n, 3, generator=g, device=DEVICE, dtype=torch.float64)
    d = _directions(n, g)
    t_max = 0.05 + 0.45 * torch.rand(n, generator=g, device=DEVICE) if segments else math.inf
    return _ray_array(o, d, t_max)


def _camera_rays(n, seed, segments=False):
    """Jittered primary rays of a 16:9 camera at z = 3.5, row by row; as
    segments, shadow rays: from points near the unit sphere to a lamp above."""
    g = _generator(seed, 1)
    w = max(1, int(round(math.sqrt(n * 16.0 / 9.0))))
    h = (n + w - 1) // w
    k = torch.arange(n, device=DEVICE)
    jit = torch.rand(n, 2, generator=g, device=DEVICE, dtype=torch.float64)
    tan = math.tan(math.radians(20.0))
    x = (2.0 * ((k % w) + jit[:, 0]) / w - 1.0) * tan * w / h
    y = (1.0 - 2.0 * ((k // w) + jit[:, 1]) / h) * tan
    d = torch.stack([x, y, torch.full_like(x, -1.0)], 1)
    d = d / d.norm(dim=1, keepdim=True)
    o = torch.tensor([0.0, 0.0, 3.5], device=DEVICE, dtype=torch.float64).expand(n, 3)
    if not segments:
        return _ray_array(o, d, math.inf)
    b = (o * d).sum(1)
    disc = (b * b - (o * o).sum(1) + 1.1025).clamp_min(0.0)  # the sphere of radius 1.05
    p = o + (-b - disc.sqrt())[:, None] * d
    lamp = torch.rand(n, 3, generator=g, device=DEVICE, dtype=torch.float64) - 0.5
    lamp[:, 1] = 2.5
    to = lamp - p
    dist = to.norm(dim=1)
    return _ray_array(p, to / dist[:, None], dist.float())


def _sphere_tris(n, seed):
    sc = scenes.displaced_icosphere(freq=int(round(math.sqrt(n / 20.0))), seed=int(seed) + 1)
    t = sc["vertices"][sc["indices"][:-2].astype(np.int64)].reshape(-1, 9)  # without its lamp
    return torch.from_numpy(np.ascontiguousarray(t, np.float32)).to(DEVICE)


def _query_inputs(case, seed):
    segments = case["op"] == "any"
    if case["shape"] == "sphere":
        return _sphere_tris(case["tris"], seed), _camera_rays(case["rays"], seed, segments)
    return _soup(case["tris"], seed), _random_rays(case["rays"], seed, segments)


def _two_level_inputs(case, seed):
    """Meshes of soup in the unit cube, random affine instances over
    [-3, 3]^3, rays aimed at them."""
    meshes = [_soup(case["tris"], seed, 2 + k) for k in range(case["meshes"])]
    mesh, m = workloads.instances_random(case["instances"], case["meshes"], int(seed) + 5)
    g = _generator(seed, 1)
    o = 8.0 * torch.rand(case["rays"], 3, generator=g, device=DEVICE, dtype=torch.float64) - 4.0
    d = 6.0 * torch.rand(case["rays"], 3, generator=g, device=DEVICE, dtype=torch.float64) - 3.0 - o
    dist = d.norm(dim=1)
    t_max = dist.float() if case["op"] == "any" else math.inf
    return meshes, mesh, m, _ray_array(o, d / dist[:, None], t_max)


def _hits(n):
    h = torch.zeros(n, 2, dtype=torch.int32, device=DEVICE)
    return Buffer(h), {"id": h[:, 0], "t": h.view(torch.float32)[:, 1]}


def _scene(case, seed):
    w, h = case["width"], case["height"]
    if case["scene"] == "cornell":
        return scenes.cornell(w, h)
    if case["scene"] == "sphere":
        return scenes.displaced_icosphere(freq=case["freq"], seed=int(seed) + 1, width=w, height=h)
    return scenes.instanced_field(w, h, n_meshes=3, freq=case["freq"], grid=5, seed=int(seed) + 1)


def _batch_jobs(case, seed):
    """(scene description, settings) of each image: meshes and images from full
    size down by factors of 1.6 and 1.3, then one instanced scene."""
    jobs = []
    for k in range(case["meshes"] + 1):
        side = max(16, int(case["side"] / 1.3 ** k))
        if k < case["meshes"]:
            f = max(7, int(case["freq"] / 1.6 ** k))
            sc = scenes.displaced_icosphere(freq=f, seed=int(seed) + 10 * k + 1, width=side, height=side)
        else:
            sc = scenes.instanced_field(side, side, n_meshes=2, freq=max(7, case["freq"] // 4), grid=4,
                                        seed=int(seed) + 3)
        jobs.append((sc, {"width": side, "height": side, "spp": case["spp"] + k, "depth": case["depth"],
                          "seed": int(seed) + k}))
    return jobs


def _film(case, seed):
    """Per-pixel sums of a finished render: exposures over four decades, dark
    pixels among them."""
    g = _generator(seed, 0)
    n = (case["height"], case["width"], 3)
    x = torch.exp(4.0 * torch.rand(n, generator=g, device=DEVICE) * math.log(10.0)) * 1e-3 * case["spp"]
    return torch.where(torch.rand(n, generator=g, device=DEVICE) < 0.05, torch.zeros_like(x), x).contiguous()


def prepare(case, seed):
    lbvh.init()
    kind = case["kind"]
    s = {"case": case}
    if kind in ("build", "refit"):
        tris, n = _soup(case["tris"], seed), case["rays"]
        s["rays"], (s["hits"], s["out"]) = Buffer(_random_rays(n, seed)), _hits(n)
        s["bvh"] = lbvh.GpuBvh()
        if kind == "refit":
            s["rest"] = Buffer(tris)
            torch.cuda.synchronize()
            s["bvh"].build_triangles_device(s["rest"], case["tris"])
            tris = _moved(tris, seed)
        s["tris"] = Buffer(tris)
    elif kind == "query":
        tris, rays = _query_inputs(case, seed)
        s["tris"], s["rays"] = Buffer(tris), Buffer(rays)
        if case["op"] == "closest":
            s["hits"], s["out"] = _hits(len(rays))
        else:
            occ = torch.zeros(len(rays), dtype=torch.uint8, device=DEVICE)
            s["hits"], s["out"] = Buffer(occ), {"occluded": occ}
        s["bvh"] = lbvh.GpuBvh()
        torch.cuda.synchronize()
        s["bvh"].build_triangles_device(s["tris"], len(tris))
        s["n_tris"] = len(tris)
    elif kind == "contacts":
        tris = _soup(case["tris"], seed)
        s["tree"] = lbvh.GpuBvh()
        s["stream"] = _shared_stream()
        s["raw"] = ctypes.c_void_p(s["stream"].cuda_stream)
        if case["op"] == "cross":
            s["tris"] = Buffer(tris)
            torch.cuda.synchronize()
            s["tree"].build_triangles_device(s["tris"], len(tris), stream=s["raw"])
            moving = _soup(case["boxes"], seed, 3, per=case["tris"])
            s["moving"] = lbvh.GpuBvh()
            s["max"] = 4 * case["boxes"] + 1024
        else:
            moving = tris
            s["max"] = 2 * case["tris"] + 1024
        s["boxes"] = Buffer(_boxes(moving))
        s["ids"] = Buffer(torch.arange(len(moving), dtype=torch.int32, device=DEVICE))
        s["pairs"] = Buffer(torch.full((s["max"], 2), -1, dtype=torch.int32, device=DEVICE))
        s["found"] = Buffer(torch.zeros(1, dtype=torch.int32, device=DEVICE))
    elif kind == "two_level":
        meshes, mesh, m, rays = _two_level_inputs(case, seed)
        tris = torch.cat(meshes).cpu().numpy()
        offsets = np.arange(case["meshes"] + 1, dtype=np.int32) * case["tris"]
        s["scene"] = two_level.TwoLevelScene(tris, offsets, two_level.make_instances(mesh, m, tris, offsets))
        s["rays"] = Buffer(rays)
        if case["op"] == "closest":
            h = torch.zeros(len(rays), 6, dtype=torch.int32, device=DEVICE)
            f = h.view(torch.float32)
            s["hits"] = Buffer(h)
            s["out"] = {"id": h[:, 0], "t": f[:, 1], "u": f[:, 2], "v": f[:, 3], "instance": h[:, 4], "local": h[:, 5]}
        else:
            occ = torch.zeros(len(rays), dtype=torch.uint8, device=DEVICE)
            s["hits"], s["out"] = Buffer(occ), {"occluded": occ}
    elif kind == "render":
        s["scene"] = render.Scene(_scene(case, seed))
        s["film"] = Buffer(torch.zeros(case["height"], case["width"], 3, device=DEVICE))
        s["seed"] = int(seed)
    elif kind == "batch":
        jobs = _batch_jobs(case, seed)
        s["scenes"] = [render.Scene(sc) for sc, _ in jobs]
        s["jobs"] = [j for _, j in jobs]
        s["films"] = [Buffer(torch.zeros(j["height"], j["width"], 3, device=DEVICE)) for j in s["jobs"]]
    else:
        s["film"] = Buffer(_film(case, seed))
        shape = (case["height"], case["width"], 3)
        kindof = torch.uint8 if case["format"] == "ppm" else torch.float32
        s["pixels"] = Buffer(torch.zeros(shape, dtype=kindof, device=DEVICE))
    torch.cuda.synchronize()
    return s


_STREAM = []


def _shared_stream():
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


# ---- one pass --------------------------------------------------------------------
def _closest(s, n_tris):
    abi.call("lux_hip_trace_closest_device", s["bvh"].handle, s["tris"].ptr, n_tris, s["rays"].ptr,
             s["case"]["rays"], s["hits"].ptr, None)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "build":
        s["bvh"].build_triangles_device(s["tris"], case["tris"])
        _closest(s, case["tris"])
        return s["out"]
    if kind == "refit":
        s["bvh"].refit_triangles_device(s["tris"], case["tris"])
        _closest(s, case["tris"])
        return s["out"]
    if kind == "query":
        if case["op"] == "closest":
            _closest(s, s["n_tris"])
        else:
            abi.call("lux_hip_trace_any_device", s["bvh"].handle, s["tris"].ptr, s["n_tris"], s["rays"].ptr,
                     case["rays"], s["hits"].ptr, None)
        return s["out"]
    if kind == "contacts":
        n = len(s["ids"].tensor)
        if case["op"] == "cross":
            s["moving"].build_device(s["boxes"], s["ids"], n, stream=s["raw"])
            abi.call("lux_hip_overlap_cross_device", s["tree"].handle, s["moving"].handle, s["max"], s["pairs"].ptr,
                     s["found"].ptr, s["raw"])
        else:
            s["tree"].build_device(s["boxes"], s["ids"], n, stream=s["raw"])
            abi.call("lux_hip_overlap_self_device", s["tree"].handle, s["max"], s["pairs"].ptr, s["found"].ptr,
                     s["raw"])
        with torch.cuda.stream(s["stream"]):  # a list in a fixed order, as a solver wants it
            pairs = torch.sort(s["pairs"].tensor.view(torch.int64).view(-1)).values
        return {"pairs": pairs, "found": s["found"].tensor}
    if kind == "two_level":
        op = s["scene"].intersect_device if case["op"] == "closest" else s["scene"].occluded_device
        op(s["rays"], case["rays"], s["hits"])
        return s["out"]
    if kind == "render":
        s["scene"].render_device(s["film"], case["width"], case["height"], case["spp"], case["depth"],
                                 seed=s["seed"])
        return s["film"].tensor
    if kind == "batch":
        render.batch_render_device(s["scenes"], s["jobs"], s["films"])
        return [f.tensor for f in s["films"]]
    to = film.ppm_pixels_device if case["format"] == "ppm" else film.pfm_pixels_device
    to(s["film"], case["width"], case["height"], case["spp"], s["pixels"])
    return s["pixels"].tensor


# ---- what a pass cannot do without -----------------------------------------------
def _walk(tris):
    """Operations of one ray through a balanced tree: both boxes of each level
    (18 each) and two triangles (50 each)."""
    return 36.0 * max(1.0, math.log2(max(2, tris))) + 100.0


def work(case):
    kind = case["kind"]
    if kind in ("build", "refit"):
        n, r = case["tris"], case["rays"]
        # triangles in, 2 n - 1 nodes of 32 bytes out, rays in, hits out
        return {"bytes": 100.0 * n + 40.0 * r, "flops": 30.0 * n + r * _walk(n)}
    if kind == "query":
        n, r = case["tris"], case["rays"]
        return {"bytes": 100.0 * n + r * (40.0 if case["op"] == "closest" else 33.0), "flops": r * _walk(n)}
    if kind == "contacts":
        n = case["tris"]
        q = case["boxes"] if case["op"] == "cross" else n
        return {"bytes": 64.0 * n + (28.0 + 64.0) * q + 8.0 * q, "flops": q * (30.0 + 12.0 * math.log2(max(2, n)))}
    if kind == "two_level":
        n, r = case["meshes"] * case["tris"], case["rays"]
        return {"bytes": 100.0 * n + 160.0 * case["instances"] + r * (56.0 if case["op"] == "closest" else 33.0),
                "flops": r * (_walk(case["instances"]) + 2 * _walk(case["tris"]))}
    if kind == "render":
        paths = float(case["width"] * case["height"] * case["spp"])
        n = 36 if case["scene"] == "cornell" else 20 * case["freq"] ** 2
        # about half of the bounces are reached; 300 operations of shading each
        return {"bytes": 12.0 * case["width"] * case["height"] + 150.0 * n,
                "flops": paths * 0.5 * (case["depth"] + 1) * (_walk(n) + 300.0)}
    if kind == "batch":
        b = f = 0.0
        for k in range(case["meshes"] + 1):
            side, n = max(16, int(case["side"] / 1.3 ** k)), 20 * max(7, int(case["freq"] / 1.6 ** k)) ** 2
            b += 12.0 * side * side + 150.0 * n
            f += side * side * (case["spp"] + k) * 0.5 * (case["depth"] + 1) * (_walk(n) + 300.0)
        return {"bytes": b, "flops": f}
    px = 3.0 * case["width"] * case["height"]
    return {"bytes": px * (5.0 if case["format"] == "ppm" else 8.0), "flops": px * 4.0}


def tolerance(case):
    """Queries, contacts and film bytes are whole numbers or single correctly
    rounded steps in a stated order (hit ids and distances are those of the
    host LBVH, bit for bit). Films depend on how sinf, cosf and powf round.
    Four times what the same renders by the CPU restatement with the host's
    libm differ by: Cornell box 5e-8 (largest pixel 6e-6); meshes with glass and
    glossy materials 3.2e-4 (0.083), where a rounding sends single paths
    another way."""
    if case["kind"] == "render" and case["scene"] == "cornell":
        return {"rel": 2e-7, "max": 2.4e-5}
    if case["kind"] in ("render", "batch"):
        return {"rel": 1.3e-3, "max": 0.33}
    return "exact"


# ---- 64-bit references -------------------------------------------------------------
def _first_hit(tris, rays, any_hit=False):
    """Closest t per ray (inf: none) by testing every triangle, in float64: the
    quantities of Moller-Trumbore as products of Pluecker coordinates."""
    t = tris.double().view(-1, 3, 3)
    v0, e1, e2 = t[:, 0], t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    r = rays.double()
    out = torch.full((len(r),), math.inf, dtype=torch.float64, device=r.device)
    step = max(1, int(1.5e8) // max(1, len(t)))
    # a = -d.n; u a = (d x e2).(o - v0); v a = -(d x e1).(o - v0); t a = n.(o - v0)
    w2, w1, w0 = torch.linalg.cross(e2, v0), torch.linalg.cross(e1, v0), (nrm * v0).sum(1)
    for b in range(0, len(r), step):
        o, d = r[b:b + step, 0:3], r[b:b + step, 3:6]
        m = torch.linalg.cross(o, d)
        a = -(d @ nrm.T)
        u = (m @ e2.T - d @ w2.T) / a
        bad = (u < 0) | (u > 1) | (a.abs() < 1e-7)
        v = (d @ w1.T - m @ e1.T) / a
        bad |= (v < 0) | (u + v > 1)
        del u, v
        tt = (o @ nrm.T - w0) / a
        bad |= ~(tt > r[b:b + step, 6:7]) | ~(tt < r[b:b + step, 7:8])
        out[b:b + step] = tt.masked_fill_(bad, math.inf).amin(1)
    return out


def _affordable(tris, rays):
    return float(tris) * float(rays) <= 1e11


def _two_level_exact(case, seed):
    meshes, mesh, m, rays = _two_level_inputs(case, seed)
    r = rays.double()
    best = torch.full((len(r),), math.inf, dtype=torch.float64, device=r.device)
    for k, mat in zip(mesh, m):
        inv = torch.linalg.inv(torch.from_numpy(mat.astype(np.float64)).to(r.device))
        q = r.clone()
        q[:, 0:3] = r[:, 0:3] @ inv[:3, :3].T + inv[:3, 3]
        q[:, 3:6] = r[:, 3:6] @ inv[:3, :3].T
        best = torch.minimum(best, _first_hit(meshes[int(k)], q))
    return best


def _pcg(state, inc):
    """PCG32 on int64 tensors: (32 output bits, next state)."""
    def shr(x, k):
        return (x >> k) & ((1 << (64 - k)) - 1)
    xs = shr(shr(state, 18) ^ state, 27) & 0xFFFFFFFF
    rot = shr(state, 59)
    out = ((xs >> rot) | (xs << ((32 - rot) & 31))) & 0xFFFFFFFF
    return out, state * 6364136223846793005 + inc


def _cornell_exact(case, seed):
    """The Cornell box path traced in float64 with the renderer's sample
    stream: Lambert walls, next-event estimation with MIS, Russian roulette."""
    sc = scenes.cornell(case["width"], case["height"])
    w, h, spp, depth = case["width"], case["height"], case["spp"], case["depth"]

    def dev(x):
        return torch.from_numpy(np.asarray(x)).to(DEVICE)

    tri = dev(sc["vertices"]).double()[dev(sc["indices"].astype(np.int64))]
    v0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    cr = torch.linalg.cross(e1, e2)
    nrm, area = cr / cr.norm(dim=1, keepdim=True), 0.5 * cr.norm(dim=1)
    mats = dev(sc["materials"]).double()[dev(sc["material_ids"].astype(np.int64))]
    albedo, emission = mats[:, 1:4], mats[:, 4:7]
    lights = torch.nonzero(emission.amax(1) > 0).view(-1)  # two triangles of equal power
    eps = 1e-5
    cam = sc["camera"].astype(np.float64)
    origin = torch.tensor(cam[0:3], device=DEVICE)
    fwd = torch.tensor(cam[3:6] - cam[0:3], device=DEVICE)
    fwd = fwd / fwd.norm()
    right = torch.linalg.cross(torch.tensor([0.0, 1.0, 0.0], device=DEVICE, dtype=torch.float64), fwd)
    right = right / right.norm()
    up = torch.linalg.cross(fwd, right)
    vh = 2.0 * math.tan(math.radians(float(cam[6])) / 2.0)
    hor, ver = right * (vh * float(cam[7])), up * vh
    low = origin + fwd - 0.5 * hor - 0.5 * ver

    n = w * h * spp
    k = torch.arange(n, device=DEVICE)
    pixel, sample = k % (w * h), k // (w * h)
    base = int(seed)
    inc = (((base >> 1) ^ (sample * 2891336453 + pixel)) << 1) | 1
    _, st = _pcg(torch.zeros_like(inc), inc)
    st = st + base + pixel * 747796405 + sample
    _, st = _pcg(st, inc)
    rng = {"s": st}

    def uniform(which):
        bits, nxt = _pcg(rng["s"], inc)
        rng["s"] = torch.where(which, nxt, rng["s"])
        return (bits >> 8).double() / float(1 << 24)

    every = torch.ones(n, dtype=torch.bool, device=DEVICE)
    jx, jy = uniform(every), uniform(every)
    for _ in range(3):
        uniform(every)
    s = ((pixel % w) + jx) / w
    t = ((h - 1 - pixel // w) + jy) / h
    d = low + s[:, None] * hor + t[:, None] * ver - origin
    d = d / d.norm(dim=1, keepdim=True)
    o = origin.expand(n, 3)

    def hits(o, d, t_max, skip=None):
        best = torch.full((n,), math.inf, dtype=torch.float64, device=DEVICE)
        prim = torch.full((n,), -1, dtype=torch.int64, device=DEVICE)
        for i in range(len(tri)):
            hh = torch.linalg.cross(d, e2[i].expand(n, 3))
            a = hh @ e1[i]
            f = 1.0 / a
            q0 = o - v0[i]
            u = f * (q0 * hh).sum(1)
            q = torch.linalg.cross(q0, e1[i].expand(n, 3))
            v = f * (d * q).sum(1)
            tt = f * (q @ e2[i])
            ok = (a.abs() >= 1e-7) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (tt > eps) & (tt < t_max)
            if skip is not None:
                ok &= skip != i
            ok &= tt < best
            best, prim = torch.where(ok, tt, best), torch.where(ok, torch.full_like(prim, i), prim)
        return best, prim

    L = torch.zeros(n, 3, dtype=torch.float64, device=DEVICE)
    T = torch.ones_like(L)
    alive, prev, prev_pdf = every.clone(), o.clone(), torch.ones(n, dtype=torch.float64, device=DEVICE)
    for bounce in range(depth + 1):
        tt, prim = hits(o, d, torch.full((n,), math.inf, dtype=torch.float64, device=DEVICE))
        alive &= prim >= 0
        i = prim.clamp_min(0)
        p, ng, wo = o + d * tt.clamp_max(1e30)[:, None], nrm[i], -d
        cos = (ng * wo).sum(1)
        lit = alive & (emission[i].amax(1) > 0) & (cos > 1e-7)
        to = p - prev
        d2 = (to * to).sum(1)
        lpdf = 0.5 / area[i] * d2 * d2.sqrt() / -(ng * to).sum(1)
        mis = torch.ones_like(cos) if bounce == 0 else prev_pdf ** 2 / (prev_pdf ** 2 + lpdf ** 2)
        L = torch.where(lit[:, None], L + T * emission[i] * mis[:, None], L)
        alive &= (albedo[i].amax(1) > 0) & (bounce < depth)
        sel = uniform(alive)
        uniform(alive)
        lu0, lu1 = uniform(alive), uniform(alive)
        j = lights[(sel.clamp_max(0.99999994) * 2).long()]
        su = lu0.sqrt()
        lp = v0[j] + (su * (1 - lu1))[:, None] * e1[j] + (su * lu1)[:, None] * e2[j]
        to = lp - p
        d2 = (to * to).sum(1)
        wi = to / d2.sqrt()[:, None]
        cl = -(nrm[j] * wi).sum(1)
        pl = 0.5 / area[j] * d2 / cl.clamp_min(1e-30)
        cs = (ng * wi).sum(1)
        side = cos * cs > 0
        see = alive & side & (cl > 1e-7) & (d2 > eps * eps)
        so = p + torch.where((cs >= 0)[:, None], ng, -ng) * eps
        to = lp - so
        dist = to.norm(dim=1)
        see &= dist > eps
        _, block = hits(so, to / dist[:, None], dist - eps, skip=prim)
        see &= block < 0
        pb = cs.abs() / math.pi
        add = albedo[i] / math.pi * emission[j] * (cs.abs() / pl * pl ** 2 / (pl ** 2 + pb ** 2))[:, None]
        L = torch.where(see[:, None], L + T * add, L)
        u0, u1 = uniform(alive), uniform(alive)
        nn = torch.where((cos < 0)[:, None], -ng, ng)
        axis = torch.zeros_like(nn)
        big = nn[:, 0].abs() > 0.9
        axis[:, 2], axis[:, 0] = big.double(), (~big).double()
        tx = torch.linalg.cross(axis, nn)
        tx = tx / tx.norm(dim=1, keepdim=True)
        ty = torch.linalg.cross(nn, tx)
        rad, phi = u0.sqrt(), 2 * math.pi * u1
        wi = (rad * phi.cos())[:, None] * tx + (1 - u0).clamp_min(0).sqrt()[:, None] * nn + (rad * phi.sin())[:, None] * ty
        wi = wi / wi.norm(dim=1, keepdim=True)
        c = (ng * wi).sum(1)
        alive &= (c.abs() > 0) & (c * cos > 0)
        nT = T * albedo[i]
        if bounce > 2:
            rr = nT.amax(1).clamp_max(0.95)
            alive &= uniform(alive) <= rr
            nT = nT / rr[:, None]
        T = torch.where(alive[:, None], nT, T)
        prev, prev_pdf = p, c.abs() / math.pi
        o, d = p + torch.where((c >= 0)[:, None], ng, -ng) * eps, wi
    return L.view(spp, h, w, 3).sum(0)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("build", "refit"):
        if not _affordable(case["tris"], case["rays"]):
            return None
        tris = _soup(case["tris"], seed)
        if kind == "refit":
            tris = _moved(tris, seed)
        return {"id": None, "t": _first_hit(tris, _random_rays(case["rays"], seed))}
    if kind == "query":
        if case["op"] == "any" or not _affordable(case["tris"], case["rays"]):
            return None
        return {"id": None, "t": _first_hit(*_query_inputs(case, seed))}
    if kind == "two_level":
        if case["op"] == "any" or not _affordable(case["instances"] * case["tris"], case["rays"]):
            return None
        none = dict.fromkeys(("id", "u", "v", "instance", "local"))
        return dict(none, t=_two_level_exact(case, seed))
    if kind == "render":
        # other scenes: a path's choices are discrete, and a 64-bit renderer of
        # every material over a mesh without a tree takes minutes
        if case["scene"] != "cornell" or case["width"] * case["height"] * case["spp"] > 1 << 20:
            return None
        return _cornell_exact(case, seed)
    if kind == "film" and case["format"] == "pfm":
        return _film(case, seed).double().flip(0) * (1.0 / case["spp"])
    return None  # whole numbers (pairs, bytes), or a batch of scenes as above
