"""The work that users of the rasterizer have it do, as cases to be timed.

Each case is one pass of a program's loop through the public Python entry
points: the reference's per-call loop, whole frames on one buffer, many views
or frames per launch, query batches, scene preparation (QuadDecomposition,
SAH batching, bake) and a training step of the draw-order model.  Scenes are
the repository's own kinds (scenes.py): boxes, a city on terrain, icosphere
instances on terrain.  A scene is the asset a program has loaded, so it is
built once per process; cameras, query boxes, meshes to prepare and training
samples come from the seed.
"""

from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from rasterizer_amd import Mlp, Rasterizer, Views, learn, scenes

FOV = math.pi / 3


def listed():
    return [
        # The reference's own frame loop, call by call: one queryVisibility per
        # occluder deciding the next rasterize, then readBackDepth for display.
        dict(name="loop_boxes_720p", kind="loop", boxes=1024, width=1280, height=720),
        # A small scene on a buffer of odd size; statuses, query bits and the
        # raw buffer all go back to the host.
        dict(name="frame_boxes_1000x600", kind="frame_host", boxes=1003, width=1000, height=600, queries=4099),
        # One frame at a time at 1080p with queries and answers in device
        # memory: the latency of a game's frame.
        dict(name="frame_city_1080p", kind="frame", terrain=512, grid=64, width=1920, height=1080, queries=65536),
        # One 4K frame of a scene of many small occluders.
        dict(name="frame_spheres_4k", kind="frame_spheres", instances=12000, width=3840, height=2160, queries=16384),
        # Frames in flight, each in the reference's query-gated loop, sorted
        # front to back on the device from each frame's eye.
        dict(name="views_city_20", kind="views", views=20, terrain=512, grid=64, width=1920, height=1080,
             queries=65536, order="eye"),
        # Many frames in flight, occluder orders known before (a replay).
        dict(name="views_city_128", kind="views", views=128, terrain=512, grid=64, width=1920, height=1080,
             queries=65536, order="sorted"),
        # The same with each frame's occluders ordered by the trained model.
        dict(name="views_city_32_learned", kind="views", views=32, terrain=512, grid=64, width=1920, height=1080,
             queries=16384, order="model"),
        # Many views of mixed size in one launch (cameras, shadow maps).
        dict(name="views_mixed_64", kind="mixed", views=64, boxes=40000, queries=16384),
        # A large batch of boxes against a finished buffer.
        dict(name="queries_city_1m", kind="queries", terrain=512, grid=64, width=1920, height=1080, queries=1000003),
        # Loading a mesh: QuadDecomposition, SAH batches and bake.
        dict(name="prepare_mesh_city", kind="mesh", terrain=512, grid=64),
        # Quads of a scene built at run time: SAH batches and bake.
        dict(name="prepare_quads_boxes", kind="quads", boxes=40000),
        # Training the draw-order model: forward and backward of one step's
        # 32 frames of 768 batches, 256 pairs each.
        dict(name="train_order_24k", kind="train", samples=24576, pairs=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng):
    """A buffer size: multiples of 8, mostly no multiple of a tile."""
    return 8 * _log_int(rng, 40, 240), 8 * _log_int(rng, 22, 135)


def draw(rng):
    kind = rng.choice(["loop", "frame_host", "frame", "frame_spheres", "views", "views", "mixed", "queries", "mesh",
                       "quads", "train"])
    w, h = _size(rng)
    terrain = rng.choice([96, 200, 333, 512])
    city = dict(terrain=terrain, grid=max(4, terrain // 8), width=w, height=h)
    if kind == "loop":
        return dict(kind=kind, boxes=_log_int(rng, 64, 4096), width=w, height=h)
    if kind == "frame_host":
        return dict(kind=kind, boxes=_log_int(rng, 64, 8000), width=w, height=h, queries=_log_int(rng, 100, 100000))
    if kind == "frame":
        return dict(kind=kind, queries=_log_int(rng, 100, 200000), **city)
    if kind == "frame_spheres":
        return dict(kind=kind, instances=_log_int(rng, 500, 12000), width=2 * w, height=2 * h,
                    queries=_log_int(rng, 100, 65536))
    if kind == "views":
        return dict(kind=kind, views=_log_int(rng, 2, 64), queries=_log_int(rng, 100, 65536),
                    order=rng.choice(["eye", "sorted", "model"]), **city)
    if kind == "mixed":
        return dict(kind=kind, views=_log_int(rng, 3, 64), boxes=rng.choice([5000, 14001, 40000]),
                    queries=_log_int(rng, 100, 16384))
    if kind == "queries":
        return dict(kind=kind, queries=_log_int(rng, 1000, 1000000), **city)
    if kind == "mesh":
        n = _log_int(rng, 24, 500)
        return dict(kind=kind, terrain=n, grid=max(2, n // rng.choice([6, 8, 13])))
    if kind == "quads":
        return dict(kind=kind, boxes=_log_int(rng, 30, 40000))
    samples = _log_int(rng, 300, 24000)
    return dict(kind=kind, samples=samples, pairs=max(1, samples // rng.choice([2, 3, 5])))


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _owner():
    """The program's context that uploads occluders for its views."""
    return Rasterizer(64, 64)


def _boxes_quads(centers, half):
    """Outward-facing quads of axis-aligned boxes, (6 n, 4, 4) float32."""
    unit = scenes.box_quads(np.zeros(3), np.ones(3))[None, :, :, :3].astype(np.float32)
    out = np.ones((centers.shape[0], 6, 4, 4), np.float32)
    out[..., :3] = centers[:, None, None, :] + unit * half[:, None, None, :]
    return out.reshape(-1, 4, 4)


def _random_boxes(rng, n, cube, lo, hi):
    c = rng.uniform(-cube, cube, (n, 3)).astype(np.float32)
    return c, np.exp(rng.uniform(math.log(lo), math.log(hi), (n, 3))).astype(np.float32)


@functools.lru_cache(maxsize=4)
def _box_scene(n):
    """n boxes at the density of 1,024 in a cube of half edge 50."""
    cube = 50.0 * (n / 1024.0) ** (1.0 / 3.0)
    c, h = _random_boxes(np.random.default_rng(1), n, cube, 0.5, 5.0)
    return _owner().prepare_scene_device(_boxes_quads(c, h)), cube


def _city_mesh(terrain, grid, seed):
    """grid^2 box buildings on a terrain^2 heightfield as one indexed mesh."""
    rng = np.random.default_rng(seed)
    hf = scenes.Heightfield(terrain, 2.0, 20.0, seed=int(rng.integers(1 << 60)))
    tri, verts = scenes.heightfield_triangles(hf)
    pitch = (terrain - 1) * 2.0 / grid
    foot = min(4.0, 0.25 * pitch)
    i, j = np.meshgrid(np.arange(grid), np.arange(grid), indexing="ij")
    cx, cz = (i.ravel() + 0.5) * pitch, (j.ravel() + 0.5) * pitch
    base = np.min([hf.height(cx + a * foot, cz + b * foot) for a in (-1, 0, 1) for b in (-1, 0, 1)], axis=0) - 1.0
    tall = np.exp(rng.uniform(math.log(5.0), math.log(80.0), grid * grid))
    centers = np.stack([cx, base + 0.5 * tall, cz], axis=1)
    halves = np.stack([np.full_like(cx, foot), 0.5 * tall, np.full_like(cx, foot)], axis=1)
    box_tri, box_verts = scenes.box_mesh(np.zeros(3), np.ones(3))
    bv = np.ones((grid * grid, box_verts.shape[0], 4), np.float32)
    bv[..., :3] = centers[:, None, :] + box_verts[None, :, :3] * halves[:, None, :]
    first = verts.shape[0] + np.arange(grid * grid)[:, None, None] * box_verts.shape[0]
    tri = np.concatenate([tri, (box_tri[None] + first).reshape(-1, 3).astype(np.uint32)])
    return hf, pitch, centers, halves, tri, np.concatenate([verts, bv.reshape(-1, 4)])


@functools.lru_cache(maxsize=5)
def _city(terrain, grid):
    hf, pitch, centers, halves, tri, verts = _city_mesh(terrain, grid, 1)
    return dict(occluders=_owner().prepare_mesh_device(tri, verts), hf=hf, pitch=pitch, grid=grid,
                extent=(terrain - 1) * 2.0, centers=centers, halves=halves)


@functools.lru_cache(maxsize=4)
def _spheres(instances):
    """Icosphere instances (80 triangles, one occluder each) on 2 km of terrain."""
    rng = np.random.default_rng(5)
    extent = 2000.0
    hf = scenes.Heightfield(128, extent / 127, 20.0, seed=77)
    tri, verts = scenes.heightfield_triangles(hf)
    occ = _owner().prepare_mesh_device(tri, verts)
    v, f = scenes.icosphere()
    scale = np.exp(rng.uniform(math.log(0.5), math.log(10.0), instances))
    px, pz = rng.uniform(0.0, extent, instances), rng.uniform(0.0, extent, instances)
    centers = np.stack([px, hf.height(px, pz) + scale, pz], axis=1)
    ang = rng.uniform(0.0, 2.0 * math.pi, instances)
    rot = np.zeros((instances, 3, 3))
    rot[:, 0, 0] = rot[:, 2, 2] = np.cos(ang)
    rot[:, 0, 2], rot[:, 2, 0] = np.sin(ang), -np.sin(ang)
    rot[:, 1, 1] = 1.0
    p = np.einsum("nij,tkj->ntki", rot * scale[:, None, None], v[f]) + centers[:, None, None, :]
    q = np.ones((instances, 80, 4, 4), np.float32)
    q[:, :, :3, :3] = p
    q[:, :, 3, :3] = p[:, :, 0]
    lo, hi = q.min(axis=(1, 2)), q.max(axis=(1, 2))
    occ = occ + _owner().bake_device(list(q.reshape(instances, -1, 4)), list(lo), list(hi))
    return dict(occluders=occ, hf=hf, extent=extent, centers=centers, scale=scale)


# ---------------------------------------------------------------------------
# Cameras and query boxes
# ---------------------------------------------------------------------------
def _mvp(eye, d, w, h):
    up = (0.0, 1.0, 0.0) if abs(d[1]) < 0.95 else (1.0, 0.0, 0.0)
    return scenes.view_projection(eye, d, up, FOV, w / h)


def _walk(city, rng, frames, w, h):
    """Eyes and matrices of a walk along one of the city's streets at eye
    height 2, a camera turning slowly."""
    g, pitch = city["grid"], city["pitch"]
    cross = float(rng.integers(1, max(2, g))) * pitch
    along = rng.uniform(0.1, 0.6) * city["extent"] + 0.5 * np.arange(frames)
    along = np.minimum(along, city["extent"] - 1.0)
    x, z = (along, np.full(frames, cross)) if rng.random() < 0.5 else (np.full(frames, cross), along)
    heading = rng.uniform(0.0, 2.0 * math.pi) + 0.01 * np.arange(frames)
    eyes = np.stack([x, city["hf"].height(x, z) + 2.0, z], axis=1).astype(np.float32)
    mvps = []
    for k in range(frames):
        d = np.array([math.cos(heading[k]), -0.08, math.sin(heading[k])])
        mvps.append(_mvp(eyes[k], d / np.linalg.norm(d), w, h))
    return eyes, mvps


def _city_queries(city, rng, n):
    """Half as many buildings as fit in a sixteenth of the batch, the rest
    props on the terrain."""
    nb = min(city["centers"].shape[0], max(1, n // 16))
    pick = rng.permutation(city["centers"].shape[0])[:nb]
    x, z = rng.uniform(0.0, city["extent"], n - nb), rng.uniform(0.0, city["extent"], n - nb)
    half = np.exp(rng.uniform(math.log(0.25), math.log(1.5), (n - nb, 3)))
    props = np.stack([x, city["hf"].height(x, z) + half[:, 1], z], axis=1)
    return scenes.aabb_bounds(np.concatenate([city["centers"][pick], props]).astype(np.float32),
                              np.concatenate([city["halves"][pick], half]).astype(np.float32))


def _front_to_back(occluders, eye):
    return [occluders[i] for i in scenes.front_to_back(occluders, eye)]


class _Buffer:
    """A torch tensor's memory as the device-pointer entry points take it."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _device_queries(boxes):
    n = boxes.shape[0]
    return (_Buffer(torch.from_numpy(boxes).cuda()), _Buffer(torch.zeros(n, dtype=torch.uint8, device="cuda")),
            _Buffer(torch.zeros(n, dtype=torch.uint8, device="cuda")))


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("loop", "frame_host"):
        occ, cube = _box_scene(case["boxes"])
        eye = rng.uniform(-0.3 * cube, 0.3 * cube, 3).astype(np.float32)
        d = rng.normal(size=3) * np.array([1.0, 0.3, 1.0])
        s["R"] = Rasterizer(case["width"], case["height"])
        s["mvp"] = _mvp(eye, d / np.linalg.norm(d), case["width"], case["height"])
        s["occluders"] = _front_to_back(occ, eye)
        s["R"].handle_array(s["occluders"])  # uploads them
        if kind == "frame_host":
            c, h = _random_boxes(rng, case["queries"], cube, 0.1, 2.0)
            s["queries"] = scenes.aabb_bounds(c, h)
    elif kind in ("frame", "queries"):
        city = _city(case["terrain"], case["grid"])
        eyes, mvps = _walk(city, rng, 1, case["width"], case["height"])
        s["R"], s["mvp"] = Rasterizer(case["width"], case["height"]), mvps[0]
        s["n"] = len(city["occluders"])
        s["handles"] = s["R"].handle_array(_front_to_back(city["occluders"], eyes[0]))
        s["boxes"], s["visible"], s["clip"] = _device_queries(_city_queries(city, rng, case["queries"]))
        torch.cuda.synchronize()
        if kind == "queries":
            s["R"].clear()
            s["R"].setModelViewProjection(s["mvp"])
            s["R"].draw_frame_handles(s["handles"], s["n"])
            s["R"].sync()
    elif kind == "frame_spheres":
        sc = _spheres(case["instances"])
        x, z = rng.uniform(0.3, 0.7, 2) * sc["extent"]
        eye = np.array([x, float(sc["hf"].height(x, z)) + 2.0, z], np.float32)
        ang = rng.uniform(0.0, 2.0 * math.pi)
        d = np.array([math.cos(ang), -0.05, math.sin(ang)])
        s["R"] = Rasterizer(case["width"], case["height"])
        s["mvp"] = _mvp(eye, d / np.linalg.norm(d), case["width"], case["height"])
        s["occluders"] = _front_to_back(sc["occluders"], eye)
        s["n"], s["handles"] = len(s["occluders"]), s["R"].handle_array(s["occluders"])
        pick = rng.integers(0, case["instances"], case["queries"])
        jitter = rng.normal(scale=5.0, size=(case["queries"], 3)) * np.array([1.0, 0.1, 1.0])
        s["boxes"], s["visible"], s["clip"] = _device_queries(scenes.aabb_bounds(
            (sc["centers"][pick] + jitter).astype(np.float32), np.repeat(sc["scale"][pick, None], 3, 1).astype(np.float32)))
        torch.cuda.synchronize()
    elif kind == "views":
        city = _city(case["terrain"], case["grid"])
        n, w, h = case["views"], case["width"], case["height"]
        eyes, mvps = _walk(city, rng, n, w, h)
        V = s["V"] = Views(_owner(), [(w, h)] * n)
        # The configuration that Views.autotune picks for these sizes.
        V.set_config(8, 0, 16 if n >= 64 else 8)
        V.set_query_gated(True)
        for k in range(n):
            V.set_occluders(k, city["occluders"] if case["order"] == "eye" else _front_to_back(city["occluders"], eyes[k]))
            V.set_queries(k, _city_queries(city, rng, case["queries"]))
        s["mvps"], s["eyes"] = mvps, eyes if case["order"] == "eye" else None
        if case["order"] == "model":
            s["model"] = learn.load(learn.WEIGHTS.with_name("order_mlp_city.npz"))
            V.set_model(s["model"], by_occluder=True)
        run(s)  # builds the plan that the program's steps replay
    elif kind == "mixed":
        occ, cube = _box_scene(case["boxes"])
        sizes = [scenes.CONFIG3_SIZES[k % 64] for k in rng.permutation(64)[:case["views"]]]
        V = s["V"] = Views(_owner(), sizes)
        V.set_config(8, 0, 8)
        s["mvps"], s["eyes"] = [], None
        for k, (w, h) in enumerate(sizes):
            eye = rng.uniform(-0.8 * cube, 0.8 * cube, 3).astype(np.float32)
            d = rng.normal(size=3)
            s["mvps"].append(_mvp(eye, d / np.linalg.norm(d), w, h))
            # 1k to all of the scene's quads, 366 to an occluder on average
            quads = math.exp(rng.uniform(math.log(1000.0), math.log(5.0 * case["boxes"])))
            sub = [occ[i] for i in rng.permutation(len(occ))[: max(1, int(quads / 366))]]
            V.set_occluders(k, _front_to_back(sub, eye))
            c = eye + rng.uniform(-50.0, 50.0, (case["queries"], 3)).astype(np.float32)
            half = np.exp(rng.uniform(math.log(0.1), math.log(2.0), (case["queries"], 3))).astype(np.float32)
            V.set_queries(k, scenes.aabb_bounds(c, half))
        run(s)
    elif kind == "mesh":
        s["R"] = _owner()
        s["tri"], s["verts"] = _city_mesh(case["terrain"], case["grid"], seed)[4:]
        s["room"] = -(-s["tri"].shape[0] // 8)
    elif kind == "quads":
        s["R"] = _owner()
        cube = 50.0 * (case["boxes"] / 1024.0) ** (1.0 / 3.0)
        s["quads"] = _boxes_quads(*_random_boxes(rng, case["boxes"], cube, 0.5, 5.0))
        s["room"] = -(-s["quads"].shape[0] // 8)
    else:
        s["x"], s["pairs"], params, norm = _training(case, seed)
        s["m"] = Mlp(seed=1)
        s["m"].set_params(params, norm)
    return s


def _training(case, seed):
    """A step's samples (features of drawn batches), ranked pairs and Glorot
    weights with the features' normalisation."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    x = rng.random((n, 16), np.float32)
    for k in (1, 5, 9, 10):  # log2 of areas, distances and labels
        x[:, k] *= 10.0
    x[:, 6] = np.round(x[:, 6])
    x[:, 11:14] = 2.0 * x[:, 11:14] - 1.0
    pairs = rng.integers(0, n, (case["pairs"], 2)).astype(np.uint32)
    params = np.zeros(Mlp.N_PARAMS, np.float32)
    at = 0
    for rows, cols in ((16, 64), (64, 64), (64, 1)):
        a = math.sqrt(6.0 / (rows + cols))
        params[at:at + rows * cols] = rng.uniform(-a, a, rows * cols)
        params[at + rows * cols:at + rows * cols + cols] = rng.uniform(-0.1, 0.1, cols)
        at += rows * cols + cols
    norm = np.concatenate([x.mean(0), 1.0 / x.std(0)]).astype(np.float32)
    return x, pairs, params, norm


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "loop":
        R = s["R"]
        R.clear()
        R.setModelViewProjection(s["mvp"])
        drawn = np.zeros(len(s["occluders"]), np.uint8)
        for k, o in enumerate(s["occluders"]):
            visible, clip = R.queryVisibility(o.m_boundsMin, o.m_boundsMax)
            if visible:
                R.rasterize(o, clip)
                drawn[k] = 2 if clip else 1
        return {"drawn": drawn, "depth": R.readBackDepth()}
    if kind == "frame_host":
        R = s["R"]
        R.clear()
        R.setModelViewProjection(s["mvp"])
        status = R.draw_frame(s["occluders"])
        visible, clip = R.query_batch(s["queries"])
        depth, hiz = R.raw()
        return {"status": status, "visible": visible.view(np.uint8), "clip": clip.view(np.uint8),
                "depth": depth.view(np.int16), "hiz": hiz.view(np.int16)}
    if kind in ("frame", "frame_spheres"):
        R = s["R"]
        R.clear()
        R.setModelViewProjection(s["mvp"])
        R.draw_frame_handles(s["handles"], s["n"])
    if kind in ("frame", "frame_spheres", "queries"):
        s["R"].query_batch_device(s["boxes"].tensor.shape[0], s["boxes"], s["visible"], s["clip"])
        return {"visible": s["visible"].tensor, "clip": s["clip"].tensor}
    if kind in ("views", "mixed"):
        V = s["V"]
        for k, m in enumerate(s["mvps"]):
            V.set_mvp(k, m)
        if s["eyes"] is not None:
            for k, e in enumerate(s["eyes"]):
                V.set_eye(k, e)
        V.run()
        V.sync()
        answers = [V.queries(k) for k in range(len(s["mvps"]))]
        return {"visible": np.concatenate([a for a, _ in answers]).view(np.uint8),
                "clip": np.concatenate([b for _, b in answers]).view(np.uint8)}
    if kind in ("mesh", "quads"):
        occ = s["R"].prepare_mesh_device(s["tri"], s["verts"]) if kind == "mesh" else s["R"].prepare_scene_device(s["quads"])
        # The set as a program stores it, in arrays with room for the largest.
        cap = s["room"]
        packets, quads, bounds = np.zeros(32 * cap, np.int32), np.zeros(cap, np.int32), np.zeros((cap, 3, 4), np.float32)
        at = 0
        for k, o in enumerate(occ):
            packets[at:at + o.packets.size] = o.packets.view(np.int32)
            at += o.packets.size
            quads[k] = o.quad_count
            bounds[k, 0], bounds[k, 1], bounds[k, 2] = o.m_boundsMin, o.m_boundsMax, o.m_center
        return {"packets": packets, "quads": quads, "bounds": bounds}
    grad, loss = s["m"].gradients(s["x"], s["pairs"])
    return {"grad": grad, "loss": np.array([loss], np.float32)}


# ---------------------------------------------------------------------------
# work, exact
# ---------------------------------------------------------------------------
def _frame_bytes(quads, w, h):
    """16 bytes a quad, depth and hiZ written once, a matrix."""
    return 16 * quads + 2 * w * h + 2 * (w // 8) * (h // 8) + 64


def _city_size(case):
    tri = 2 * (case["terrain"] - 1) ** 2 + 12 * case["grid"] ** 2
    return tri, case["terrain"] ** 2 + 8 * case["grid"] ** 2


def work(case):
    kind = case["kind"]
    flops = 0
    if kind == "loop":
        # readBackDepth writes 4 bytes a pixel
        b = _frame_bytes(6 * case["boxes"], case["width"], case["height"]) + 4 * case["width"] * case["height"]
    elif kind == "frame_host":
        b = 2 * _frame_bytes(6 * case["boxes"], case["width"], case["height"]) + 34 * case["queries"]
    elif kind in ("frame", "views"):
        b = _frame_bytes(_city_size(case)[0] // 2, case["width"], case["height"]) + 34 * case["queries"]
        b *= case.get("views", 1)
    elif kind == "frame_spheres":
        b = _frame_bytes(80 * case["instances"] + 127 ** 2, case["width"], case["height"]) + 34 * case["queries"]
    elif kind == "mixed":
        # the mean of the views' sizes and of their quads
        px = sum(w * h for w, h in scenes.CONFIG3_SIZES) / 64
        quads = 5.0 * case["boxes"] / math.log(5.0 * case["boxes"] / 1000.0)
        b = case["views"] * (16 * quads + 2 * px + px / 32 + 64 + 34 * case["queries"])
    elif kind == "queries":
        b = 34 * case["queries"] + 2 * case["width"] * case["height"]
    elif kind == "mesh":
        tri, verts = _city_size(case)
        b = 12 * tri + 16 * verts + 16 * (tri // 2)
    elif kind == "quads":
        b = (64 + 16) * 6 * case["boxes"]
    else:
        b = 64 * case["samples"] + 8 * case["pairs"] + 8 * Mlp.N_PARAMS
        flops = 3 * 10368 * case["samples"]
    return {"bytes": float(b), "flops": float(flops)}


def exact(case, seed):
    """Loss and gradient of a training step in 64 bits (the other cases give
    whole numbers, or values chosen from their inputs)."""
    if case["kind"] != "train":
        return None
    x, pairs, params, norm = _training(case, seed)
    t = torch.from_numpy(params).double().requires_grad_()
    n = torch.from_numpy(norm).double()
    w1, b1, w2, b2, w3, b3 = torch.split(t, [1024, 64, 4096, 64, 64, 1])
    h = (torch.from_numpy(x).double() - n[:16]) * n[16:]
    h = torch.nn.functional.gelu(h @ w1.view(16, 64) + b1)
    h = torch.nn.functional.gelu(h @ w2.view(64, 64) + b2)
    score = h @ w3 + b3
    p = torch.from_numpy(pairs.astype(np.int64))
    loss = torch.nn.functional.softplus(score[p[:, 1]] - score[p[:, 0]]).mean()
    loss.backward()
    return {"grad": t.grad.numpy(), "loss": loss.detach().reshape(1).numpy()}
