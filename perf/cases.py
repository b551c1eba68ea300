"""The calls a user of raytrace_amd makes, for timing: single frames to host and
to device memory, batches, the serving loop, scenes loaded and edited, and the
reference's own RayTracer::start.

A case names its kind, its scene and its sizes; listed() are the fixed ones,
draw() gives others of the same ranges.  prepare() builds the scene through the
Scene API from the seed and makes it resident, as a program does before it
renders; run() is one pass through the public entry points.

Scenes (all seeded): "spheres", a plane and spheres placed here; "mesh", the
displaced icosphere with 64 spheres; "soup" and "field", the triangle soup and
the height field of the batch workload; "terrain", the refraction workload's
terrain with 256 sphere meshes and 4 samples per pixel.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import raytrace_amd as rt
from raytrace_amd import _capi

NORMAL_MODE = 0x3  # the reference's primary-only normal view


def listed():
    return [
        # A thumbnail request rendered alone: the smallest size of the request
        # stream, where launches and latency are everything.
        {"name": "thumbnail", "kind": "frame", "scene": "field", "tris": 10000, "lights": 2, "width": 64, "height": 64,
         "level": 2, "spp": 1, "ids": False, "device": False},
        # The plane-and-spheres frame of the first workload, with primary ids
        # and hit distances back in host memory (picking, depth compositing).
        {"name": "spheres", "kind": "frame", "scene": "spheres", "tris": 0, "lights": 2, "width": 640, "height": 480,
         "level": 3, "spp": 1, "ids": True, "device": False},
        # The headline frame: 1080p, depth 4, 200,000 triangles, into device memory.
        {"name": "frame_1080p", "kind": "frame", "scene": "mesh", "tris": 200000, "lights": 4, "width": 1920,
         "height": 1080, "level": 4, "spp": 1, "ids": False, "device": True},
        # An antialiased frame of a ragged size (no multiple of any block) to the host.
        {"name": "ragged_4spp", "kind": "frame", "scene": "soup", "tris": 34385, "lights": 3, "width": 801, "height": 451,
         "level": 3, "spp": 4, "ids": False, "device": False},
        # Branching ray trees: refraction, depth 8, 16 lights, 4 samples; the
        # largest amount of rays here.
        {"name": "refraction", "kind": "frame", "scene": "terrain", "tris": 784898, "lights": 16, "width": 960,
         "height": 540, "level": 8, "spp": 4, "ids": False, "device": True},
        # A primary-only normal view, as an editor shows while the user moves.
        {"name": "normal_view", "kind": "frame", "scene": "mesh", "tris": 200000, "lights": 4, "width": 1280,
         "height": 720, "level": 0, "spp": 1, "ids": False, "device": False, "mode": NORMAL_MODE},
        # Sixty requests of the mixed request stream over eight resident scenes, one batch.
        {"name": "batch_mixed", "kind": "batch", "requests": 60, "scenes": 8, "largest": 1024, "stream": 3},
        # A dozen thumbnails of odd sizes over two scenes: a batch bound by its launches.
        {"name": "batch_thumbs", "kind": "batch", "requests": 12, "scenes": 2, "largest": 96, "stream": 4},
        # A burst of requests that all wait when the serving loop starts.
        {"name": "serve_burst", "kind": "serve", "requests": 32, "scenes": 4, "largest": 320, "stream": 5},
        # A scene loaded (upload and BVH build), its first frame rendered, and released.
        {"name": "load_scene", "kind": "load", "scene": "mesh", "tris": 200000, "lights": 4, "width": 480, "height": 270,
         "level": 2},
        # A resident scene edited between frames: an object moved (BVH refit), a
        # light moved (shading tables), both back (refit), a frame after each.
        {"name": "edit_scene", "kind": "edit", "scene": "mesh", "tris": 50000, "lights": 4, "width": 320, "height": 180,
         "level": 2},
        # The reference's RayTracer::start, twice on one tracer, as its viewer calls it.
        {"name": "drop_in", "kind": "drop_in", "scene": "mesh", "tris": 20480, "lights": 2, "width": 768, "height": 576,
         "level": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "serve", "load", "edit", "drop_in"])
    if kind in ("batch", "serve"):
        largest = _log_int(rng, 65, 1024 if kind == "batch" else 512)
        return {"kind": kind, "requests": _log_int(rng, 2, 60), "scenes": rng.randint(1, 8), "largest": largest,
                "stream": rng.randrange(1 << 20)}
    scene = rng.choice(["spheres", "mesh", "soup", "field", "terrain"] if kind == "frame" else ["mesh", "soup", "field"])
    case = {"kind": kind, "scene": scene, "tris": _log_int(rng, 1000, 500000 if kind == "frame" else 250000),
            "lights": rng.randint(1, 6), "width": _log_int(rng, 33, 1920), "height": _log_int(rng, 33, 1080),
            "level": rng.randint(0, 5)}
    if scene == "spheres":
        case["tris"] = 0
    if scene == "terrain":
        case["tris"] = 784898
        case["lights"] = rng.randint(1, 16)
        case["width"], case["height"] = min(case["width"], 960), min(case["height"], 540)
        case["level"] = rng.randint(1, 8)
    if kind != "frame":
        case["width"], case["height"] = min(case["width"], 1280), min(case["height"], 720)
        return case
    case |= {"spp": rng.choice([1, 1, 4]), "ids": rng.random() < 0.4, "device": rng.random() < 0.4}
    if case["spp"] == 4:
        case["width"], case["height"] = min(case["width"], 960), min(case["height"], 540)
    option = rng.choice(["plain", "plain", "plain", "fp64_retest", "megakernel", "normal_view"])
    if option == "fp64_retest" and scene != "terrain":
        case["retest"] = True
    if option == "megakernel" and scene != "terrain":
        case["mega"] = True
        case["width"], case["height"] = min(case["width"], 640), min(case["height"], 480)
    if option == "normal_view":
        case["mode"] = NORMAL_MODE
    return case


# ---- scenes ---------------------------------------------------------------


def _spheres_numbers(seed, lights):
    """The seeded numbers of the "spheres" scene: [(radius, centre, kd, ks)], [light position]."""
    g = np.random.default_rng(1000 + seed)
    f = np.float32
    balls = [(f(g.uniform(0.3, 1.5)), g.uniform(-5, 5, 3).astype(f), g.uniform(0, 1, 3).astype(f), f(g.uniform(0, 1)))
             for _ in range(8)]
    return balls, [g.uniform((-8, 4, -8), (8, 12, 8)).astype(f) for _ in range(lights)]


def _spheres(seed, lights, width, height):
    balls, lamps = _spheres_numbers(seed, lights)
    hs = rt.HostScene.new()
    hs.resize(width, height)
    hs.set_env_light((0.05, 0.05, 0.05, 1.0))
    hs.add_plane()
    for r, c, kd, ks in balls:
        n = hs.add_sphere(float(r))
        hs.set_position(n, (*c.tolist(), 1.0))
        hs.set_material(n, (0.2 * kd).tolist(), kd.tolist(), (float(ks),) * 3, 32.0, reflect=0.3)
    for p in lamps:
        n = hs.add_light(2, (0.15, 0.55, 0.3), (0.0, 0.0, 1.0, 256.0))
        hs.set_light_position(n, (*p.tolist(), 1.0))
    return hs


def _host_scene(case, seed):
    name, size = case["scene"], dict(width=case["width"], height=case["height"], n_lights=case["lights"])
    s = 1 + seed % (1 << 30)
    if name == "spheres":
        return _spheres(seed, case["lights"], case["width"], case["height"])
    if name == "mesh":
        return rt.HostScene.workload(2, seed=s, detail=max(2, round(math.sqrt(case["tris"] / 20))), **size)
    if name == "terrain":
        return rt.HostScene.workload(5, seed=s, detail=4, **size)
    return rt.HostScene.workload(3, seed=s, index=0 if name == "soup" else 1, detail=case["tris"], **size)


_stream = None  # the program's render stream


def _render_stream():
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _requests(case):
    """[(scene, width, height)] of the case's requests, sides up to `largest`."""
    g = np.random.default_rng(case["stream"])
    n, top = case["requests"], case["largest"]
    w = np.round(33 * (top / 33) ** g.random(n)).astype(int)
    h = np.round(33 * (0.75 * top / 33) ** g.random(n)).astype(int)
    return [(int(g.integers(case["scenes"])), int(a), int(b)) for a, b in zip(w, h)]


# ---- the calls ------------------------------------------------------------


def prepare(case, seed):
    rt.init(0)
    kind = case["kind"]
    if kind in ("batch", "serve"):
        hs = [rt.HostScene.workload(3, seed=1 + seed % (1 << 30), index=i) for i in range(case["scenes"])]
        ds = [rt.DeviceScene(h) for h in hs]
        reqs = _requests(case)
        items = [(ds[s], rt.params(w, h, max_level=hs[s].info.max_level)) for s, w, h in reqs]
        state = {"kind": kind, "scenes": (hs, ds), "items": items}
        if kind == "batch":
            state["out"] = [{"rgb": np.zeros((h, w, 3), np.uint8), "ids": None} for _, w, h in reqs]
        return state
    W, H = case["width"], case["height"]
    hs = _host_scene(case, seed)
    state = {"kind": kind, "host": hs, "level": case["level"]}
    if kind == "drop_in":
        return state
    state["params"] = rt.params(
        W, H, max_level=case["level"], spp=case.get("spp", 1), seed=seed,
        engine=rt.RTG_ENGINE_MEGAKERNEL if case.get("mega") else rt.RTG_ENGINE_AUTO,
        flags=rt.RTG_FLAG_FP64_RETEST if case.get("retest") else 0, mode=case.get("mode", rt.RTG_MODE_RAYTRACE))
    if kind != "load":
        state["scene"] = rt.DeviceScene(hs)
    if kind == "edit":
        g = np.random.default_rng(seed)
        state["num"] = 0
        state["places"] = [(*g.uniform(-1.5, 1.5, 3).tolist(), 1.0), (*g.uniform(-1.5, 1.5, 3).tolist(), 1.0)]
        state["lamps"] = [(*g.uniform((-8, 4, -8), (8, 12, 8)).tolist(), 1.0) for _ in range(2)]
        hs.set_position(0, state["places"][0])
        hs.set_light_position(0, state["lamps"][0])
        state["scene"].update(hs)
    if kind == "frame":
        state["device"], state["ids"] = case["device"], case["ids"]
        if case["device"]:
            new = lambda shape, dtype: torch.zeros(shape, dtype=dtype, device="cuda:0")
            state["rgb"] = new((H, W, 3), torch.uint8)
            state["counts"] = new((4,), torch.int64)
            if case["ids"]:
                state["ids_out"], state["t_out"] = new((H, W, 2), torch.int32), new((H, W), torch.float32)
            _render_stream().wait_stream(torch.cuda.current_stream())
        else:
            state["out"] = {"rgb": np.zeros((H, W, 3), np.uint8),
                            "ids": np.zeros((H, W, 2), np.int32) if case["ids"] else None,
                            "t": np.zeros((H, W), np.float32) if case["ids"] else None}
    return state


def _frame_device(state):
    at = lambda a: C.c_void_p(a.data_ptr()) if a is not None else None
    p = state["params"]
    rc = _capi.load().rtg_render_device(state["scene"].h, C.byref(p), at(state["rgb"]), at(state.get("ids_out")),
                                        at(state.get("t_out")), at(state["counts"]),
                                        C.c_void_p(_render_stream().cuda_stream))
    _capi.check(rc, "rtg_render_device")
    return {k: state[k] for k in ("rgb", "ids_out", "t_out", "counts") if k in state}


def run(state):
    kind = state["kind"]
    if kind == "frame":
        if state["device"]:
            return _frame_device(state)
        out = state["scene"].render(state["params"], ids=state["ids"], tprim=state["ids"], out=state["out"])
        return {k: out[k] for k in ("rgb", "ids", "t") if out[k] is not None}
    if kind == "batch":
        outs, _ = rt.render_batch(state["items"], ids=False, out=state["out"])
        return [o["rgb"] for o in outs]
    if kind == "serve":
        outs, _, _ = rt.serve([(d, p, 0.0) for d, p in state["items"]])
        return outs
    if kind == "drop_in":
        return state["host"].raytrace(max_level=state["level"], frames=2)[0]
    hs, p = state["host"], state["params"]
    frame = lambda ds: ds.render(p, ids=False, tprim=False)["rgb"]
    if kind == "load":
        ds = rt.DeviceScene(hs)
        rgb = frame(ds)
        ds.close()
        return rgb
    ds, frames = state["scene"], []
    for place, lamp in ((1, 0), (1, 1), (0, 0)):
        hs.set_position(state["num"], state["places"][place])
        hs.set_light_position(0, state["lamps"][lamp])
        ds.update(hs)
        frames.append(frame(ds))
    return frames


def work(case):
    """Every triangle's record read once (128 B each where it is uploaded, 120 B of
    primitive and shading data where it is resident), every output written once;
    per ray a descent of a binary tree, 20 operations a box, and a primitive test."""
    kind = case["kind"]
    if kind in ("batch", "serve"):
        side = lambda top: (top - 33) / math.log(top / 33)  # mean of the log-uniform sides
        pixels = case["requests"] * side(case["largest"]) * side(max(34, 0.75 * case["largest"]))
        tris = 144000 * case["scenes"]  # mean of the batch scenes' 1k .. 1M
        rays, out, per_tri = pixels * 5, pixels * 3, 120
    else:
        tris, per_tri, frames = case["tris"] + 64, 120, {"edit": 3, "drop_in": 2}.get(kind, 1)
        pixels = case["width"] * case["height"] * frames
        lit = 0 if case.get("mode") else case["lights"]
        rays = pixels * case.get("spp", 1) * (1 + lit)
        out = pixels * (15 if case.get("ids") else 3)
        if kind in ("load", "drop_in"):
            per_tri = 128 + 120
        if kind == "edit":
            per_tri = 128 * 2 + 120
    return {"bytes": float(tris * per_tri + out), "flops": float(rays * (20 * 2 * math.log2(tris + 2) + 40))}


# ---- 64-bit values --------------------------------------------------------


def exact(case, seed):
    """Primary hit distances of the plane-and-spheres scene at one sample per
    pixel, in 64 bits; no values for bytes, ids and counts, and none for the
    triangle scenes (a scan of every triangle for every pixel)."""
    if case["kind"] != "frame" or case["scene"] != "spheres" or not case["ids"] or case["spp"] != 1:
        return None
    W, H = case["width"], case["height"]
    balls, _ = _spheres_numbers(seed, case["lights"])
    # the default camera: at (0, 4, 15), looking along -z, 45 degrees high
    o = np.array([0.0, 4.0, 15.0])
    dp = math.tan(45.0 * math.pi / 360) / (H // 2)
    x, y = (np.arange(W) - W // 2) * dp, (np.arange(H) - H // 2) * dp
    d = np.stack(np.broadcast_arrays(x[None, :], y[:, None], -1.0), -1)
    d = d / np.linalg.norm(d, axis=-1, keepdims=True)
    t = np.full((H, W), 1e20)
    # the default plane: through the origin, facing up
    down = d[..., 1] < -1e-6
    t[down] = -o[1] / d[..., 1][down]
    for r, c, _, _ in balls:
        s = o - c.astype(np.float64)
        b = d @ s
        disc = b * b - s @ s + float(r) ** 2
        hit = (disc >= 0) & (b <= 0)
        near = -(b + np.sqrt(np.where(hit, disc, 0.0)))
        t = np.where(hit & (near > 1e-6) & (near < t), near, t)
    if case["device"]:
        return {"rgb": None, "ids_out": None, "t_out": t, "counts": None}
    return {"rgb": None, "ids": None, "t": t}
