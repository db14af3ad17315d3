"""A scene whose nodes take more than 4 GB: its kernels' 64-bit node addresses
against the kernels that count (exact node test, 64-bit throughout) and, for
the batch, against a batch of one."""
import ctypes as C
import sys

import numpy as np
import pytest

import ptamd
from helpers import PyScene

pytestmark = pytest.mark.gpu

COUNT, DIRECT, SORT = ptamd.PT_FLAG_COUNT_TRAVERSAL, ptamd.PT_FLAG_DIRECT, ptamd.PT_FLAG_MATERIAL_SORT
CACHE = ptamd.PT_FLAG_RADIANCE_CACHE
MESHES, SIDE = 52, 1448  # height fields of 2 x 1448^2 triangles each


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def field():
    x, z = np.meshgrid(np.linspace(0, 10, SIDE + 1, dtype=np.float32), np.linspace(0, 10, SIDE + 1, dtype=np.float32))
    v = np.stack([x, 0.4 * np.sin(3 * x) * np.cos(2 * z), z], 2).reshape(-1, 3)
    q = (np.arange(SIDE, dtype=np.uint32)[:, None] * (SIDE + 1) + np.arange(SIDE, dtype=np.uint32)[None]).ravel()
    f = np.concatenate([np.stack([q, q + SIDE + 1, q + 1], 1), np.stack([q + 1, q + SIDE + 1, q + SIDE + 2], 1)])
    return np.ascontiguousarray(v), np.ascontiguousarray(f)


def wide_scene(field, media):
    """One height field as 52 meshes (52 structures), each an instance at its
    own place, under a light; with `media` also a volume and a cylinder."""
    s = PyScene()
    mats = [s.lambert((0.7, 0.6, 0.5)), s.material(ptamd.PT_MAT_METAL, s.texture((0.8, 0.8, 0.8)), params=(0.2,)),
            s.material(ptamd.PT_MAT_OREN_NAYAR, s.texture((0.4, 0.6, 0.7)), params=(0.3,))]
    glow = s.material(ptamd.PT_MAT_DIFFUSE_LIGHT, s.texture((6, 6, 6)))
    for k in range(MESHES):
        s.meshes.append((*field, None, None, mats[k % 3]))
        s.instance(ptamd.PT_GEOM_MESH, k, 0, np.hstack([np.eye(3), [[10.0 * (k % 8)], [0.3 * (k % 4)], [10.0 * (k // 8)]]]))
    s.rects.append((1, 1, 10.0, 40.0, 10.0, 30.0, 25.0, glow))
    s.instance(ptamd.PT_GEOM_RECTS, 0, 1)
    s.lights.append({"type": ptamd.PT_LIGHT_RECT, "axis": 1, "rect": (10.0, 40.0, 10.0, 30.0, 25.0), "emission": (6, 6, 6)})
    if media:
        fog = s.material(ptamd.PT_MAT_ISOTROPIC, s.texture((0.9, 0.9, 0.9)))
        s.volumes.append((ptamd.PT_VOLUME_SPHERE, (30.0, 4.0, 20.0), (5.0, 0.0, 0.0), 0.1, fog))
        s.cylinders.append(((12.0, 0.0, 12.0), 6.0, 1.5, mats[0]))
        s.instance(ptamd.PT_GEOM_VOLUMES, 0, 1)
        s.instance(ptamd.PT_GEOM_CYLINDERS, 0, 1)
    return s


def camera(W, H):
    c = ptamd.Camera()
    c.origin[:] = (30.0, 20.0, -25.0)
    c.lower_left[:] = (30.0 - 16.0, 20.0 - 24.0, -25.0 + 20.0)
    c.horizontal[:] = (32.0, 0.0, 0.0)
    c.vertical[:] = (0.0, 18.0, 0.0)
    c.u[:], c.v[:], c.w[:] = (1, 0, 0), (0, 1, 0), (0, 0, -1)
    c.time1 = 1.0
    return c


def rays_over(n):
    rng = np.random.default_rng(1)
    r = np.zeros(n, ptamd.RAY_DTYPE)
    r["org"] = rng.uniform((0, 2, 0), (80, 20, 65), (n, 3))
    r["dir"] = rng.uniform((0, -1, 0), (80, 1, 65), (n, 3)) - r["org"]
    r["tmin"], r["tmax"] = 1e-3, np.inf
    return r


@pytest.mark.parametrize("media", [False, True])
def test_nodes_beyond_4_gb(field, media):
    W, H, frames = 320, 180, 9  # 2^18 paths and more: all bounds of the launch shapes
    with ptamd.Context(0) as ctx:
        s = wide_scene(field, media)
        say(f"[gpu] {MESHES} meshes of {len(field[1])} triangles, media {media}")
        ctx.set_scene(s.desc())
        a = ctx.build_accel()
        say(f"[gpu] {a.num_nodes} nodes, {a.num_nodes * 128 / 2**32:.2f} x 4 GB, built in {a.build_ms:.0f} ms")
        assert a.num_nodes * 128 > 1 << 32
        ctx.set_camera(camera(W, H))
        rays = rays_over(200003)
        say("[gpu] queries")
        fast = ctx.trace_closest(rays)
        exact, _ = ctx.trace_closest(rays, counted=True)
        assert np.array_equal(fast.view(np.uint8), exact.view(np.uint8))
        hit = exact["inst"][exact["inst"] >= 0]
        assert np.all(np.bincount(hit, minlength=MESHES)[:MESHES] > 100)
        light = exact["inst"] == MESHES
        assert np.array_equal(ctx.trace_occluded(rays), ((exact["inst"] >= 0) & ~light).astype(np.uint8))

        def image(flags, n=frames):
            st = ctx.render(ptamd.RenderParams(W, H, 6, 1, 3, 0, flags, 0), 0, n)
            return ctx.read_accum(W, H)[0], st

        for flags in (0, SORT):
            say(f"[gpu] render, flags {flags}")
            ref, rst = image(flags | COUNT)
            for f, n in ((flags, frames), (flags | DIRECT, frames)):
                img, st = image(f, n)
                assert np.array_equal(img, ref)
                assert (st.extension_rays, st.shadow_rays) == (rst.extension_rays, rst.shadow_rays)
                assert st.node_fetches == 0 < rst.node_fetches
            ref1, _ = image(flags | COUNT, 1)  # few lanes per wave
            assert np.array_equal(image(flags, 1)[0], ref1)
        assert ref.max() > 0
        say("[gpu] batch of one")
        ptamd.render_batch([ctx], [ptamd.RenderParams(W, H, 6, 1, 3, 0, SORT, 0)], [frames], stats=False)
        assert np.array_equal(ctx.read_accum(W, H)[0], ref)
        if media:
            return
        say("[gpu] radiance cache")
        got = []
        for flags in (CACHE | SORT, CACHE | SORT | COUNT, CACHE, CACHE | COUNT):
            ctx.cache_init(3)
            ctx.render(ptamd.RenderParams(W, H, 6, 1, 3, 0, flags, 0), 0, 2)
            got.append((ctx.read_accum(W, H)[0], ctx.cache_params()))
        for k in (0, 2):
            for x, y in zip(got[k], got[k + 1]):
                assert np.array_equal(x, y)
