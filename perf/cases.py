"""What a user of the path tracer has it do, as timed cases: previews, final
renders, batches of scenes, ray queries, acceleration-structure builds and
the radiance cache, each through the public entry points of `ptamd`.

Every case is a dict of plain values; `kind` says which entry points one pass
calls:

  preview  set_camera, one frame, the displayed image (a viewer whose camera
           moves: nothing is captured, latency and launches count)
  final    every sample of one image, then its accumulation (a still)
  batch    many uneven scenes in one render_batch, then their images
  queries  trace_closest and trace_occluded of host rays (picking, visibility)
  rays     trace_closest_device on rays that are resident on the GPU
  build    set_scene, build_accel, then the first queries against it
  cached   one frame of the orbit animation with the radiance cache training
           online, then its accumulation
  network  one training step of the cache's network and an inference batch
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "optix-path-tracer_amd"))
import ptamd  # noqa: E402
from ptamd import metrics  # noqa: E402

SCENES = {"spheres": ptamd.PT_SCENE_RANDOM_SPHERES, "cornell": ptamd.PT_SCENE_CORNELL,
          "meshes": ptamd.PT_SCENE_MESHES, "moving": ptamd.PT_SCENE_MOVING_SPHERES,
          "next_week": ptamd.PT_SCENE_NEXT_WEEK}
# triangles of the mesh scene's variants 1..6 (8 octaspheres of 8 * 4^L) and
# of the full workload (variant 0: 2^20)
MESH_LEVEL = {0: 7, 1: 1, 2: 2, 3: 3, 4: 4, 5: 5, 6: 6}


def listed():
    return [
        # a thumbnail or test tile: the smallest render call, all latency
        {"name": "tile_cornell", "kind": "preview", "scene": "cornell", "variant": 0, "width": 64, "height": 64},
        # an interactive viewer on the full mesh scene
        {"name": "preview_meshes", "kind": "preview", "scene": "meshes", "variant": 0, "width": 1920, "height": 1080},
        # the sphere scene's still at its own size: few paths, 50 bounces
        {"name": "final_spheres", "kind": "final", "scene": "spheres", "variant": 0, "width": 400, "height": 267,
         "spp": 16, "graph": True},
        # the Cornell box's still at its own size: light sampling, 16 bounces
        {"name": "final_cornell", "kind": "final", "scene": "cornell", "variant": 0, "width": 512, "height": 512,
         "spp": 64, "graph": True},
        # media, boxes, a Perlin texture and a thousand-sphere group at an odd size
        {"name": "final_next_week", "kind": "final", "scene": "next_week", "variant": 0, "width": 301, "height": 203,
         "spp": 16, "graph": False},
        # the largest: a production still of the mesh scene under its HDRI
        {"name": "final_meshes", "kind": "final", "scene": "meshes", "variant": 0, "width": 1920, "height": 1080,
         "spp": 96, "graph": False},
        # every fourth scene of the 64-scene workload at its own size and samples
        {"name": "batch_16", "kind": "batch", "first": 0, "step": 4, "count": 16, "divide": 1},
        # a tool that asks for a hundred thousand rays from host memory
        {"name": "queries_host", "kind": "queries", "scene": "meshes", "variant": 0, "n": 100003},
        # a renderer that keeps its rays on the GPU
        {"name": "rays_device", "kind": "rays", "scene": "meshes", "variant": 0, "n": 4194321},
        # a scene is loaded, or a deformed one replaced
        {"name": "build_meshes", "kind": "build", "variant": 0, "n": 4096},
        # the orbit animation with the learned cache, one sample per frame
        {"name": "cached_orbit", "kind": "cached", "variant": 0, "width": 1920, "height": 1080},
        # the network by itself, at the render loop's batch
        {"name": "network", "kind": "network", "train": 16384, "infer": 65537},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, most):
    """An image size of at most `most` pixels, any aspect from 3:4 to 2:1."""
    px = _log(rng, 4096, most)
    a = rng.uniform(0.75, 2.0)
    return max(16, int(math.sqrt(px * a))), max(16, int(math.sqrt(px / a)))


def draw(rng):
    kind = rng.choice(["preview", "final", "final", "final", "batch", "queries", "rays", "build", "cached", "network"])
    scene = rng.choice(["spheres", "cornell", "meshes", "meshes", "next_week", "moving"])
    variant = rng.choice([0, 4, 5, 6]) if scene == "meshes" else 0 if scene == "cornell" else rng.randrange(8)
    if kind == "preview":
        w, h = _size(rng, 1920 * 1080)
        return {"kind": kind, "scene": scene, "variant": variant, "width": w, "height": h}
    if kind == "final":
        # up to the largest listed case's paths on the mesh scene; the other
        # scenes' paths are longer
        w, h = _size(rng, 1920 * 1080 if scene == "meshes" else 512 * 512)
        most = (1920 * 1080 * 64 if scene == "meshes" else 512 * 512 * 32) // (w * h)
        return {"kind": kind, "scene": scene, "variant": variant, "width": w, "height": h,
                "spp": _log(rng, 1, max(2, min(256, most))), "graph": rng.random() < 0.5}
    if kind == "batch":
        step = rng.choice([3, 5, 7, 9])
        return {"kind": kind, "first": rng.randrange(8), "step": step, "count": rng.randrange(2, 56 // step + 1),
                "divide": rng.choice([1, 2, 4])}
    if kind == "queries":
        return {"kind": kind, "scene": scene, "variant": variant, "n": _log(rng, 100, 1000000) | 1}
    if kind == "rays":
        return {"kind": kind, "scene": scene, "variant": variant, "n": _log(rng, 1000, 8000000) | 1}
    if kind == "build":
        return {"kind": kind, "variant": rng.choice([2, 3, 4, 5, 6]), "n": _log(rng, 100, 10000)}
    if kind == "cached":
        w, h = _size(rng, 1920 * 1080)
        return {"kind": kind, "variant": rng.choice([0, 4, 5, 6]), "width": max(w, 128), "height": max(h, 128)}
    return {"kind": kind, "train": _log(rng, 64, 65536), "infer": _log(rng, 32, 1000000)}


# ------------------------------------------------------------------ inputs
class _State(dict):
    """A case's inputs and the handles its program keeps; the contexts go
    with it."""

    def __del__(self):
        for c in self.get("ctxs", ()):
            c.close()


def _moved(cam, rs, share=0.2):
    """The scene's camera moved by a little along its own axes."""
    c = ptamd.Camera.from_buffer_copy(cam)
    f = np.linalg.norm(np.array(c.lower_left[:]) - np.array(c.origin[:]))
    a, b = rs.uniform(-share, share, 2) * f
    d = a * np.array(c.u[:]) + b * np.array(c.v[:])
    c.origin[:] = (np.array(c.origin[:]) + d).tolist()
    c.lower_left[:] = (np.array(c.lower_left[:]) + d).tolist()
    return c


def _camera(scene, name, rs):
    if name == "meshes":
        return metrics.orbit_camera(scene.info, int(rs.randint(0, 300)))
    return _moved(scene.camera, rs)


def _built(scene):
    ctx = ptamd.Context(0)
    ctx.set_scene(scene.desc)
    ctx.build_accel()
    return ctx


BOXES = {"spheres": ((-12, 0, -12), (12, 3, 12)), "cornell": ((0, 0, 0), (555, 555, 555)),
         "meshes": ((-12, -8, -12), (12, 8, 12)), "moving": ((-12, 0, -12), (12, 3, 12)),
         "next_week": ((-400, 0, -300), (600, 550, 600))}


def _rays(name, n, rs):
    """Rays between two random points of the scene's box, half of them to
    infinity and half ending at the second point (visibility)."""
    lo, hi = (np.array(b, np.float32) for b in BOXES[name])
    a = lo + rs.random_sample((n, 3)).astype(np.float32) * (hi - lo)
    b = lo + rs.random_sample((n, 3)).astype(np.float32) * (hi - lo)
    rays = np.zeros(n, ptamd.RAY_DTYPE)
    rays["org"] = a
    rays["dir"] = b - a
    rays["tmin"] = 1e-3
    rays["tmax"] = np.where(rs.random_sample(n) < 0.5, np.float32(np.inf), np.float32(1.0))
    return rays


def _bf16(x):
    """FP32 -> BF16 bit patterns (round to nearest even)."""
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(torch.bfloat16).view(torch.int16).numpy().view(
        np.uint16)


def _features(n, rs):
    """Feature rows as the renderer encodes them: sines and cosines of the
    position, directions and albedos in [0, 1], zeros from 83 on."""
    f = np.zeros((n, ptamd.PT_CACHE_INPUTS), np.float32)
    p = rs.random_sample((n, 3)).astype(np.float32)
    for a in range(3):
        for q in range(12):
            f[:, 24 * a + 2 * q] = np.sin(np.pi * 2.0**q * p[:, a])
            f[:, 24 * a + 2 * q + 1] = np.cos(np.pi * 2.0**q * p[:, a])
    f[:, 72:83] = rs.random_sample((n, 11))
    return _bf16(f)


def _parameters(rs):
    """He-uniform weights, zero biases, in the library's parameter order."""
    out = []
    for i, o in ((96, 64), (64, 64), (64, 64), (64, 64), (64, 3)):
        a = math.sqrt(6.0 / i)
        out += [rs.uniform(-a, a, i * o), np.zeros(o)]
    return np.concatenate(out).astype(np.float32)


def _network_inputs(case, seed):
    rs = np.random.RandomState(seed % (1 << 31))
    p = _parameters(rs)
    ft = _features(case["train"], rs)
    target = (rs.exponential(0.5, (case["train"], 3))).astype(np.float32)
    return p, ft, target, _features(case["infer"], rs)


def prepare(case, seed):
    rs = np.random.RandomState(seed % (1 << 31))
    kind = case["kind"]
    if kind == "network":
        p, ft, target, fi = _network_inputs(case, seed)
        ctx = ptamd.Context(0)
        ctx.cache_init(0)
        ctx.cache_params(p)
        return _State(kind=kind, ctxs=[ctx], ft=ft, target=target, fi=fi)
    if kind == "batch":
        scenes = [ptamd.Scene(ptamd.PT_SCENE_BATCH, 0, 0, case["first"] + k * case["step"]) for k in range(case["count"])]
        ctxs = [_built(s) for s in scenes]
        for c, s in zip(ctxs, scenes):
            c.set_camera(_moved(s.camera, rs))
        return _State(kind=kind, ctxs=ctxs, params=[s.render_params() for s in scenes],
                      frames=[max(1, s.info.spp // case["divide"]) for s in scenes],
                      sizes=[(s.info.width, s.info.height) for s in scenes])
    if kind == "build":
        scene = ptamd.Scene(ptamd.PT_SCENE_MESHES, 0, 0, case["variant"])
        # the vertices of a deforming scene: another seed is another shape
        for k in range(scene.desc.num_meshes):
            m = scene.desc.meshes[k]
            v = np.ctypeslib.as_array(m.vertices, (m.num_vertices, 3))
            v *= np.float32(rs.uniform(0.9, 1.1))
        return _State(kind=kind, ctxs=[ptamd.Context(0)], scene=scene, rays=_rays("meshes", case["n"], rs))
    if kind == "cached":
        scene = ptamd.Scene(ptamd.PT_SCENE_MESHES, case["width"], case["height"], case["variant"])
        ctx = _built(scene)
        ctx.cache_init(seed % 1000)
        params = scene.render_params(flags=scene.info.flags | ptamd.PT_FLAG_RADIANCE_CACHE)
        return _State(kind=kind, ctxs=[ctx], params=params, camera=_camera(scene, "meshes", rs),
                      size=(case["width"], case["height"]))
    w, h = case.get("width", 0), case.get("height", 0)
    # the mesh scene's variant is its tessellation; the others' the scene's
    # own random sequence (the Cornell box has none)
    scene = ptamd.Scene(SCENES[case["scene"]], w, h, case["variant"])
    ctx = _built(scene)
    if kind in ("preview", "final"):
        flags = scene.info.flags | (ptamd.PT_FLAG_GRAPH if case.get("graph") else 0)
        return _State(kind=kind, ctxs=[ctx], params=scene.render_params(flags=flags),
                      camera=_camera(scene, case["scene"], rs), size=(w, h), spp=case.get("spp", 1))
    rays = _rays(case["scene"], case["n"], rs)
    if kind == "queries":
        return _State(kind=kind, ctxs=[ctx], rays=rays)
    rays = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
    hits = torch.empty((case["n"], 4), dtype=torch.int32, device="cuda")
    return _State(kind=kind, ctxs=[ctx], rays=rays, hits=hits)


# ------------------------------------------------------------------- a pass
def run(s):
    kind, ctx = s["kind"], s["ctxs"][0]
    if kind == "preview":
        ctx.set_camera(s["camera"])
        ctx.render(s["params"], 0, 1, stats=False)
        return ctx.read_display(*s["size"])
    if kind == "final":
        ctx.set_camera(s["camera"])
        ctx.render(s["params"], 0, s["spp"], stats=False)
        return ctx.read_accum(*s["size"])[0]
    if kind == "batch":
        ptamd.render_batch(s["ctxs"], s["params"], s["frames"], stats=False)
        return [c.read_display(w, h) for c, (w, h) in zip(s["ctxs"], s["sizes"])]
    if kind == "queries":
        hits = ctx.trace_closest(s["rays"])
        return {"t": hits["t"], "inst": hits["inst"], "prim": hits["prim"], "occluded": ctx.trace_occluded(s["rays"])}
    if kind == "rays":
        rays, hits = s["rays"], s["hits"]
        ctx._check(ctx.lib.pt_trace_closest_device(ctx.h, C.c_void_p(rays.data_ptr()), len(rays),
                                                   C.c_void_p(hits.data_ptr())), "pt_trace_closest_device")
        ctx.sync()  # the library's own stream wrote the hits
        return {"t": hits.view(torch.float32)[:, 0], "inst": hits[:, 1], "prim": hits[:, 2]}
    if kind == "build":
        ctx.set_scene(s["scene"].desc)
        a = ctx.build_accel()
        hits = ctx.trace_closest(s["rays"])
        return {"nodes": int(a.num_nodes), "bytes": int(a.bytes), "t": hits["t"], "inst": hits["inst"],
                "prim": hits["prim"]}
    if kind == "cached":
        ctx.set_camera(s["camera"])
        ctx.render(s["params"], 0, 1, stats=False)
        return {"image": ctx.read_accum(*s["size"])[0], "params": ctx.cache_params()}
    loss, grad = ctx.cache_train(s["ft"], s["target"])
    return {"loss": loss, "grad": grad, "params": ctx.cache_params(), "y": ctx.cache_infer(s["fi"])}


# --------------------------------------------------------------------- work
# closest-hit and shadow rays per camera path, and the structure's bytes, as
# the counted passes of the benchmark give them
RAYS_PER_PATH = {"meshes": 1.8, "cornell": 5.6, "spheres": 2.7, "moving": 3.0, "next_week": 12.0}
# node visits per ray: 4 slab tests of 24 operations each, plus two to five
# primitive tests of about 50
FLOPS_PER_RAY = {"meshes": 500, "cornell": 500, "spheres": 900, "moving": 900, "next_week": 1500}


def _scene_bytes(name, variant):
    if name == "meshes":
        tris = 64 * 4 ** MESH_LEVEL[variant]
        env = 2048 * 1024 if variant == 0 else 256 * 128
        return tris * (48 + 128 / 3) + env * 16
    return {"spheres": 485 * 32, "cornell": 2048, "moving": 489 * 32, "next_week": 1500 * 40}[name]


def work(case):
    kind = case["kind"]
    if kind == "network":
        # forward, backward through the activations, weight gradients; both
        # sets of feature rows once, targets and outputs once
        flops = case["train"] * 2 * (18624 + 12480 + 18624) + case["infer"] * 2 * 18624
        return {"bytes": (case["train"] + case["infer"]) * (192 + 12) + 4 * 4 * ptamd.PT_CACHE_PARAMS, "flops": flops}
    if kind == "batch":
        paths = bytes_ = 0
        for k in range(case["count"]):
            side, spp, prims = _batch_spec(case["first"] + k * case["step"])
            paths += side * side * max(1, spp // case["divide"])
            bytes_ += side * side * (4 + 24) + prims * 90
        return {"bytes": bytes_, "flops": paths * 2.0 * 600}
    if kind == "build":
        # indices and vertices in, records and nodes out
        tris = 64 * 4 ** MESH_LEVEL[case["variant"]]
        return {"bytes": tris * (12 + 6 + 48 + 128 / 3), "flops": tris * 30}
    if kind in ("queries", "rays"):
        per = 32 + 16 if kind == "rays" else 2 * 32 + 16 + 1
        return {"bytes": case["n"] * per + _scene_bytes(case["scene"], case["variant"]),
                "flops": case["n"] * FLOPS_PER_RAY[case["scene"]] * (1 if kind == "rays" else 2)}
    scene = case.get("scene", "meshes")
    px = case["width"] * case["height"]
    out = 4 if kind == "preview" else 24
    flops = px * case.get("spp", 1) * RAYS_PER_PATH[scene] * FLOPS_PER_RAY[scene]
    return {"bytes": px * out + _scene_bytes(scene, case["variant"]), "flops": flops}


def _batch_spec(i):
    """(side, spp, primitives) of scene i of the 64-scene workload."""
    raw = np.random.RandomState(3).randint(0, 1 << 32, 3 * 64, dtype=np.uint64)
    a, b, c = ((int(x) >> 8) / 16777216.0 for x in raw[3 * i:3 * i + 3])
    prims = 50 * 100**a if i < 32 else 1e4 * 200**a
    return int(round(256 * 4**b)), (4, 16, 64)[min(2, int(3 * c))], prims


def tolerance(case):
    """Measured against a build of the same code with fused multiply-adds:
    queries are off by 3e-8 (distances) and 4e-6 (ids), the network by 3e-9
    (its operands are BF16, so a sum in another order can move a hidden unit
    by a BF16 rounding).  Images are chains of decisions: where one sample
    path in thousands takes another (a grazing hit, a light sample lit or
    not) it carries another radiance, 0.003 of a still's 2-norm, 0.01 under
    the HDRI's sun, 4e-4 of a preview's bytes."""
    kind = case["kind"]
    if kind == "network":
        return {"rel": 1e-2, "max": 0.3}
    if kind in ("queries", "rays", "build"):
        return {"rel": 2e-7, "max": 2e-5, "differ": 2e-5}
    return {"rel": 2e-2, "max": 0.9, "differ": 2e-3}


# -------------------------------------------------------------------- exact
def _exact_network(case, seed):
    p, ft, target, fi = _network_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def values(bits):
        return torch.from_numpy(bits.view(np.int16).copy()).view(torch.bfloat16).to(dev).double()

    w = torch.from_numpy(p).to(dev).double().requires_grad_(True)

    def forward(x):
        o = 0
        for k, (i, u) in enumerate(((96, 64), (64, 64), (64, 64), (64, 64), (64, 3))):
            x = x @ w[o:o + i * u].reshape(u, i).t() + w[o + i * u:o + i * u + u]
            o += i * u + u
            x = torch.relu(x) if k < 4 else x
        return x

    y = forward(values(ft))
    t = torch.from_numpy(target).to(dev).double()
    r = torch.expm1(torch.clamp(y, max=20.0))
    loss = ((r - t) ** 2 / (r.detach() ** 2 + 0.01)).sum() / len(t)
    (g,) = torch.autograd.grad(loss, w)
    with torch.no_grad():
        # Adam's first step: both moments' bias corrections cancel
        w -= 1e-3 * g / (g.abs() + 1e-8)
        out = torch.cat([forward(values(fi[k:k + (1 << 17)])) for k in range(0, len(fi), 1 << 17)])
    return {"loss": None, "grad": g.cpu(), "params": w.detach().cpu(), "y": out.cpu()}


def exact(case, seed):
    """The network in 64 bits.  A rendered image has no such value (one
    sample path is a chain of decisions), and the queries' distances are held
    to the traversal-independent closest hit by the test suite's brute-force
    checks."""
    return _exact_network(case, seed) if case["kind"] == "network" else None
