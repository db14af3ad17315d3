"""Launch-shape machinery on the GPU: batches replayed from a captured
hipGraph and the autotuned launch shape give images bit-identical to the
directly launched render (every shape traces the same paths)."""
import sys

import numpy as np
import pytest

import ptamd
from helpers import PyScene, icosphere

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    c = ptamd.Context(0)
    yield c
    c.close()


def setup(ctx, cfg, W, H, variant=0):
    sc = ptamd.Scene(cfg, W, H, variant)
    ctx.set_scene(sc.desc)
    ctx.build_accel()
    ctx.set_camera(sc.camera)
    return sc


def look_camera(origin, W, H, vfov=40.0):
    """Pinhole camera at `origin` looking at 0, up +y."""
    o = np.array(origin, np.float64)
    w = o / np.linalg.norm(o)
    u = np.cross([0, 1, 0], w)
    u /= np.linalg.norm(u)
    v = np.cross(w, u)
    hh = np.tan(np.radians(vfov) / 2)
    hw = hh * W / H
    c = ptamd.Camera()
    c.origin[:] = o
    c.lower_left[:] = o - hw * u - hh * v - w
    c.horizontal[:] = 2 * hw * u
    c.vertical[:] = 2 * hh * v
    c.u[:], c.v[:], c.w[:] = u, v, w
    return c


def image(ctx, params, f0, n):
    st = ctx.render(params, f0, n)
    acc, frames = ctx.read_accum(params.width, params.height)
    return acc, st


# 45x31: a ragged path count (2790 slots per two-frame batch)
@pytest.mark.parametrize("cfg,W,H", [(ptamd.PT_SCENE_CORNELL, 96, 64), (ptamd.PT_SCENE_MESHES, 96, 64),
                                     (ptamd.PT_SCENE_CORNELL, 45, 31)])
def test_graph_replay_is_bit_identical(ctx, cfg, W, H):
    sc = setup(ctx, cfg, W, H, 3 if cfg == ptamd.PT_SCENE_MESHES else 0)
    say(f"[gpu] graph replay scene {cfg} {W}x{H}")
    base = sc.render_params(frames_per_batch=2)
    ref, _ = image(ctx, base, 0, 7)
    g = sc.render_params(flags=sc.info.flags | ptamd.PT_FLAG_GRAPH, frames_per_batch=2)
    a, st = image(ctx, g, 0, 7)      # 3 graph replays and a direct 1-frame tail
    assert np.array_equal(a, ref)
    assert st.extend_ms == 0  # no per-kernel events inside graphs
    b, _ = image(ctx, g, 0, 7)       # replays of the cached graph
    assert np.array_equal(b, ref)
    # progressive continuation through graphs
    image(ctx, g, 0, 4)
    c2, _ = image(ctx, g, 4, 3)
    assert np.array_equal(c2, ref)


def test_autotune_picks_a_shape_with_identical_results(ctx):
    W = H = 128
    sc = setup(ctx, ptamd.PT_SCENE_CORNELL, W, H)
    say("[gpu] autotune cornell 128x128")
    p = sc.render_params()
    ref, _ = image(ctx, p, 0, 128)
    r = ctx.autotune(p, 128)
    say(f"[gpu] tuned: frames_per_batch={r.frames_per_batch} sort={r.material_sort} graph={r.graph} "
        f"{r.ms_per_frame:.3f} ms/frame over {r.candidates} candidates")
    assert r.candidates >= 4 and r.frames_per_batch >= 1 and r.ms_per_frame > 0
    t = sc.render_params(flags=p.flags | ptamd.PT_FLAG_TUNED)
    a, _ = image(ctx, t, 0, 128)
    assert np.array_equal(a, ref)


DRIVER = ptamd.REPO / "tests" / "_bin" / "facade_driver"


@pytest.mark.parametrize("scene,cfg,W,H,frames", [("Cornell", ptamd.PT_SCENE_CORNELL, 96, 80, 4),
                                                  ("RandomSpheres", ptamd.PT_SCENE_RANDOM_SPHERES, 90, 60, 3)])
def test_facade_launch_loop_equals_render(tmp_path, scene, cfg, W, H, frames):
    """The reference's main.cpp pattern through the host scene API: the
    scene function, acc_buffer / display_buffer bound as context variables,
    an empty launch that builds, then context["frame"] and
    Context::launch(0, W, H) per frame, accBuffer->map() and
    displayBuffer->map() (tests/facade_driver.cpp).  The mapped buffers
    equal one pt_render of the same frames."""
    import subprocess

    if not DRIVER.exists():
        pytest.fail("tests/_bin/facade_driver is not built (run __graft_entry__.build())")
    out = tmp_path / "maps.bin"
    say(f"[gpu] facade driver {scene} {W}x{H} x {frames}")
    subprocess.run([str(DRIVER), scene, str(W), str(H), str(frames), str(out)], check=True, timeout=120)
    raw = out.read_bytes()
    acc_map = np.frombuffer(raw[:W * H * 16], np.float32).reshape(H, W, 4)
    disp_map = np.frombuffer(raw[W * H * 16:], np.uint8).reshape(H, W, 4)
    sc = ptamd.Scene(cfg, W, H)
    with ptamd.Context(0) as ctx:
        ctx.set_scene(sc.desc)
        ctx.build_accel()
        ctx.set_camera(sc.camera)
        ctx.render(sc.render_params(), 0, frames)
        acc, n = ctx.read_accum(W, H)
        disp = ctx.read_display(W, H)
    assert n == frames
    assert np.array_equal(acc_map[..., :3], acc.astype(np.float32))
    assert np.all(acc_map[..., 3] == frames)
    assert np.array_equal(disp_map, disp)


# depths around the bounce where one launch takes over the rest of a batch
# (1, or 4 in the extended scenes from 2^18 paths on), a path count below one
# wave, and image sizes around 2^18 paths, where waves start with fewer lanes
@pytest.mark.parametrize("cfg,W,H,frames,depths", [
    (ptamd.PT_SCENE_CORNELL, 7, 5, 1, (1, 2, 3)), (ptamd.PT_SCENE_CORNELL, 96, 64, 2, (1, 2, 16)),
    (ptamd.PT_SCENE_RANDOM_SPHERES, 513, 511, 1, (1, 50)), (ptamd.PT_SCENE_CORNELL, 512, 512, 1, (1, 2, 5)),
    (ptamd.PT_SCENE_RANDOM_SPHERES, 91, 45, 1, (2, 50)), (ptamd.PT_SCENE_NEXT_WEEK, 513, 512, 1, (4, 5, 9)), (ptamd.PT_SCENE_MESHES, 61, 47, 3, (2, 12)),
    (ptamd.PT_SCENE_NEXT_WEEK, 61, 47, 2, (2, 50)), (ptamd.PT_SCENE_MOVING_SPHERES, 61, 47, 2, (3, 50))])
def test_last_bounces_in_one_launch_are_bit_identical(ctx, cfg, W, H, frames, depths):
    sc = setup(ctx, cfg, W, H, 3 if cfg == ptamd.PT_SCENE_MESHES else 0)
    flags = sc.info.flags | ptamd.PT_FLAG_KEEP_PATHS
    for depth in depths:
        say(f"[gpu] one launch for the last bounces: scene {cfg} {W}x{H} depth {depth}")
        got = []
        for extra in (0, ptamd.PT_FLAG_DIRECT):
            p = sc.render_params(flags=flags | extra)
            p.max_depth = depth
            acc, st = image(ctx, p, 0, frames)
            got.append((acc, *ctx.read_paths(W, H),
                        np.array([st.extension_rays, st.shadow_rays, st.exhausted_paths, st.nan_paths])))
        for a, b in zip(*got):
            assert np.array_equal(a, b, equal_nan=True)


def one_program_meshes():
    """Meshes and a ground rect of one Lambertian material."""
    s = PyScene()
    m = s.lambert((0.6, 0.6, 0.6))
    v, f = icosphere(4)
    s.meshes.append((v, f, None, None, m))
    rng = np.random.default_rng(0)
    for _ in range(12):
        s.instance(ptamd.PT_GEOM_MESH, 0, 0, np.hstack([np.eye(3) * rng.uniform(0.5, 1.5), rng.uniform(-5, 5, (3, 1))]))
    s.rects.append((1, 0, -50.0, 50.0, -50.0, 50.0, -6.0, m))
    s.instance(ptamd.PT_GEOM_RECTS, 0, 1)
    return s


# The bounce from which one launch runs the rest (extend_launches), on both
# sides of each of the rule's sizes, and the same image, ray counts and path
# ends as a launch per kernel and bounce gives.
@pytest.mark.parametrize("cfg,sort,W,H,frames,first", [
    (ptamd.PT_SCENE_MESHES, False, 1000, 2097, 16, 1), (ptamd.PT_SCENE_MESHES, False, 1024, 2049, 16, 4),
    (ptamd.PT_SCENE_MESHES, True, 1000, 1047, 8, 1), (ptamd.PT_SCENE_MESHES, True, 1024, 1025, 8, 4),
    ("one program", False, 1000, 1047, 4, 1), ("one program", False, 1024, 1025, 4, 4),
    (ptamd.PT_SCENE_CORNELL, True, 1000, 1047, 64, 1), (ptamd.PT_SCENE_CORNELL, True, 1024, 1025, 64, 4),
    (ptamd.PT_SCENE_RANDOM_SPHERES, False, 1024, 1025, 64, 1), (ptamd.PT_SCENE_RANDOM_SPHERES, True, 1024, 1025, 8, 4),
    (ptamd.PT_SCENE_NEXT_WEEK, True, 512, 511, 1, 1), (ptamd.PT_SCENE_NEXT_WEEK, False, 513, 512, 1, 4)])
def test_where_the_last_bounces_launch_begins(ctx, cfg, sort, W, H, frames, first):
    if cfg == "one program":
        s = one_program_meshes()
        ctx.set_scene(s.desc())
        ctx.build_accel()
        ctx.set_camera(look_camera((0.8, 1.5, 14.0), W, H))
        make = lambda flags: ptamd.RenderParams(W, H, 8, 1, 3, 0, flags, 0)  # noqa: E731
        base = 0
    else:
        sc = setup(ctx, cfg, W, H, 3 if cfg == ptamd.PT_SCENE_MESHES else 0)
        make = lambda flags: sc.render_params(flags=flags)  # noqa: E731
        base = sc.info.flags & ~ptamd.PT_FLAG_MATERIAL_SORT
    if sort:
        base |= ptamd.PT_FLAG_MATERIAL_SORT
    say(f"[gpu] last bounces of {W * H * frames} paths, scene {cfg}, sort {sort}")
    a, sa = image(ctx, make(base), 0, frames)
    b, sb = image(ctx, make(base | ptamd.PT_FLAG_DIRECT), 0, frames)
    assert sa.extend_launches == first and sa.shade_launches == first + 1
    assert sb.extend_launches == sb.shade_launches == make(base).max_depth
    assert np.array_equal(a, b)
    for k in ("extension_rays", "shadow_rays", "exhausted_paths", "nan_paths"):
        assert getattr(sa, k) == getattr(sb, k), k


# The kernels that count use the exact node test: the same hits, hence images.
@pytest.mark.parametrize("cfg,variant,W,H,frames", [
    (ptamd.PT_SCENE_RANDOM_SPHERES, 0, 400, 267, 16), (ptamd.PT_SCENE_CORNELL, 0, 256, 256, 16),
    (ptamd.PT_SCENE_MESHES, 5, 480, 270, 8), (ptamd.PT_SCENE_NEXT_WEEK, 0, 301, 203, 8),
    (ptamd.PT_SCENE_MOVING_SPHERES, 0, 301, 203, 8)])
def test_counting_kernels_render_the_same_image(ctx, cfg, variant, W, H, frames):
    sc = setup(ctx, cfg, W, H, variant)
    say(f"[gpu] default and counting image, scene {cfg}")
    a, sa = image(ctx, sc.render_params(), 0, frames)
    b, sb = image(ctx, sc.render_params(flags=sc.info.flags | ptamd.PT_FLAG_COUNT_TRAVERSAL), 0, frames)
    assert np.array_equal(a, b)
    assert (sa.extension_rays, sa.shadow_rays) == (sb.extension_rays, sb.shadow_rays)
