"""Rays that meet the conservative node test (the kernels that do not count)
at its edges, against the exact one (the kernels that count) and the oracle:
equal distances, origins in the planes of boxes, directions of any length."""
import sys

import numpy as np
import pytest

import ptamd
import ptref
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


def same(a, b):
    return (a["t"] == b["t"]) & (a["inst"] == b["inst"]) & (a["prim"] == b["prim"])


def rays_of(org, d, tmin, tmax=np.inf):
    r = np.zeros(len(org), ptamd.RAY_DTYPE)
    r["org"], r["dir"], r["tmin"], r["tmax"] = org, d, tmin, tmax
    return r


# Overlapping rects in one plane k, as one group and as instances of their
# own: every ray meets many hits at the same distance, and the smallest
# (instance, primitive) wins, however the subtrees' entry distances round.
# The padding of a flat box (1e-4) is less than the rounding of a distance
# from k = 420 on.
@pytest.mark.parametrize("k", [400.0, 555.0, 4000.0, 30000.0, 400000.0])
@pytest.mark.parametrize("mesh", [False, True])
def test_equal_distances_go_to_the_smallest_key(ctx, k, mesh):
    rng = np.random.default_rng(int(k))
    s = PyScene()
    m = s.lambert((0.5, 0.5, 0.5))

    def rect(axis):
        a, b = np.sort(rng.uniform(-100, 100, (2, 2)), axis=1)
        return (axis, 0, a[0], a[1], b[0], b[1], k, m)

    s.rects = [rect(q % 3) for q in range(600)]
    s.instance(ptamd.PT_GEOM_RECTS, 0, 300)
    for q in range(300, 600):
        s.instance(ptamd.PT_GEOM_RECTS, q, 1)
    for q in rng.permutation(300)[:60]:  # duplicates of earlier rects
        s.instance(ptamd.PT_GEOM_RECTS, 300 + int(q), 1)
    if mesh:  # the kernels for scenes with meshes (lanes take rays one after another)
        v, f = icosphere(2, 50.0, (-500.0, -500.0, -500.0))
        s.meshes.append((v, f, None, None, m))
        s.instance(ptamd.PT_GEOM_MESH, 0, 0)
    desc = s.desc()
    n = 60000
    axis = np.arange(n) % 3
    # origins at and near 0 on the facing axis, where the plane's distance
    # takes all of its rounding from the reciprocal
    org = rng.uniform(-60, 60, (n, 3))
    near = rng.choice([0.0, 1e-3, 0.3, 1.0, 7.0], n) * rng.uniform(-1, 1, n)
    org[np.arange(n), axis] = near
    to = rng.uniform(-90, 90, (n, 3))
    to[np.arange(n), axis] = k
    rays = rays_of(org, (to - org) * rng.uniform(0.1, 3.0, (n, 1)), 1e-3)
    say(f"[gpu] equal distances at {k}, meshes {mesh}: {n} rays")
    ctx.set_scene(desc)
    ctx.build_accel()
    a = ctx.trace_closest(rays)
    b, _ = ctx.trace_closest(rays, counted=True)
    o = ptref.OracleScene(desc).trace(rays, brute=True)
    assert (o["inst"] >= 0).mean() > 0.5
    assert np.array_equal(a["t"], o["t"])
    differ = ~same(a, o)
    assert not differ.any(), f"{differ.sum()} of {n} rays"
    assert same(b, o).all()


def faces_at_zero():
    """Boxes and rects with faces and edges in the planes x, y, z = 0."""
    rng = np.random.default_rng(3)
    s = PyScene()
    m = s.lambert((0.5, 0.5, 0.5))
    for q in range(96):
        lo, hi = np.sort(rng.uniform(-8, 8, (2, 3)), axis=0)
        axis = q % 3
        lo[axis], hi[axis] = (0.0, abs(hi[axis]) + 0.1) if q % 2 else (-abs(lo[axis]) - 0.1, 0.0)
        s.boxes.append((tuple(lo), tuple(hi), m))
        a, b = np.sort(rng.uniform(-8, 8, (2, 2)), axis=1)
        e = a if q % 4 < 2 else b
        e[q % 2] = 0.0
        e.sort()
        s.rects.append((axis, 0, a[0], a[1], b[0], b[1], float(rng.uniform(-8, 8)), m))
    s.instance(ptamd.PT_GEOM_BOXES, 0, 48)
    s.instance(ptamd.PT_GEOM_RECTS, 0, 48)
    for q in range(48, 96):
        s.instance(ptamd.PT_GEOM_BOXES, q, 1)
        s.instance(ptamd.PT_GEOM_RECTS, q, 1)
    return s, m


@pytest.mark.parametrize("mesh", [False, True])
def test_rays_in_the_planes_of_faces(ctx, mesh):
    """Directions with zero components from origins in a face's or an edge's
    own plane at 0, where the rounding margins of the node test are zero: such
    a ray runs along edges, which belong to the faces, and (octahedra) between
    two triangles that both have the edge."""
    rng = np.random.default_rng(4)
    s, m = faces_at_zero()
    if mesh:
        v = np.float32([[2, 0, 0], [-2, 0, 0], [0, 2, 0], [0, -2, 0], [0, 0, 2], [0, 0, -2]])
        f = np.uint32([[a, b, c] for a in (0, 1) for b in (2, 3) for c in (4, 5)])
        for q in range(8):  # a mesh each
            s.meshes.append((v * np.float32(0.2 + 0.3 * q), f, None, None, m))
            s.instance(ptamd.PT_GEOM_MESH, q, 0)
    n = 60000
    k = np.arange(n)
    org = rng.uniform(-9, 9, (n, 3))
    d = rng.normal(size=(n, 3))
    axis = rng.integers(0, 3, n)
    org[k, axis] = rng.choice([0.0, -0.0, 1e-30, -1e-30], n)
    d[k, axis] = rng.choice([0.0, -0.0], n)
    second = k[k % 3 == 0]
    d[second, (axis[second] + 1) % 3] = 0.0
    rays = rays_of(org, d, 1e-3)
    desc = s.desc()
    say(f"[gpu] rays in the planes of faces, meshes {mesh}: {n} rays")
    ctx.set_scene(desc)
    ctx.build_accel()
    a = ctx.trace_closest(rays)
    b, _ = ctx.trace_closest(rays, counted=True)
    differ = ~same(a, b)
    assert (b["inst"] >= 0).mean() > 0.3
    assert not differ.any(), f"{differ.sum()} of {n} rays"


# Directions from denormal to almost the largest length: rects, boxes and
# triangles are met whatever the length (a sphere's or cylinder's square of it
# overflows or vanishes), as long as the distance itself is a number.  The
# conservative node test may add a leaf that the exact one's rounding passes
# by, so it may only be nearer.  Below lengths of 1e-35 the spacing of denormal
# components (1.4e-45) passes 1e-3 of a rounding (6e-8), so that an instance's
# ray leaves the world's by what decides a few edges in 30000 rays; there the
# two tests only have to agree in all but 1e-3.
@pytest.mark.parametrize("exponent", [-40, -36, -33, -30, -25, -15, 15, 25, 30, 33, 36])
def test_directions_of_any_length(ctx, exponent):
    rng = np.random.default_rng(100 + exponent)
    s, m = faces_at_zero()
    v, f = icosphere(3, 3.0, (1.0, 2.0, -1.0))
    s.meshes.append((v, f, None, None, m))
    for q in range(6):
        M = np.hstack([np.diag(rng.uniform(0.3, 2.0, 3)), rng.uniform(-6, 6, (3, 1))])
        s.instance(ptamd.PT_GEOM_MESH, 0, 0, M if q else None)
    s.rects += [(q % 3, 0, -7.0, 7.0, -7.0, 7.0, float(rng.uniform(-9, 9)), m) for q in range(12)]
    s.instance(ptamd.PT_GEOM_RECTS, 96, 12)
    n = 30000
    k = np.arange(n)
    org = rng.uniform(-9, 9, (n, 3))
    unit = rng.normal(size=(n, 3))
    unit /= np.linalg.norm(unit, axis=1, keepdims=True)
    rows = k[k % 4 == 1]
    unit[rows, rng.integers(0, 3, len(rows))] = 0.0
    d = (unit * 10.0 ** (exponent + rng.uniform(-1, 1, (n, 1)))).astype(np.float32)
    desc = s.desc()
    say(f"[gpu] directions of length 1e{exponent}: {n} rays")
    ctx.set_scene(desc)
    ctx.build_accel()
    rays = rays_of(org, d, 0.0)
    a = ctx.trace_closest(rays)
    b, _ = ctx.trace_closest(rays, counted=True)
    differ = ~same(a, b)
    nearer = (a["t"] < b["t"]) | ((a["t"] == b["t"]) & ((a["inst"] < b["inst"]) |
                                                       ((a["inst"] == b["inst"]) & (a["prim"] < b["prim"]))))
    if exponent > -34:
        assert np.all(~differ | nearer), f"{(differ & ~nearer).sum()} of {n} rays"
    assert differ.mean() <= 1e-3
    assert np.array_equal(ctx.trace_occluded(rays), (a["inst"] >= 0).astype(np.uint8))
    if exponent in (-36, 33):
        assert (b["inst"] >= 0).mean() > 0.3
    # with an infinite component the distances along it are zero: a miss
    d[k, rng.integers(0, 3, n)] = rng.choice([np.inf, -np.inf], n)
    a = ctx.trace_closest(rays_of(org, d, 1e-3))
    assert np.all(a["inst"] < 0)


# Every traversal loop relies on this to end: children come after their
# parents, each node has one parent, and every leaf is one the structure owns.
@pytest.mark.parametrize("cfg,variant", [(ptamd.PT_SCENE_CORNELL, 0), (ptamd.PT_SCENE_RANDOM_SPHERES, 0),
                                         (ptamd.PT_SCENE_MESHES, 1), (ptamd.PT_SCENE_MESHES, 0),
                                         (ptamd.PT_SCENE_NEXT_WEEK, 0), (ptamd.PT_SCENE_MOVING_SPHERES, 0)])
def test_structures_are_trees(ctx, cfg, variant):
    sc = ptamd.Scene(cfg, 64, 64, variant)
    say(f"[gpu] structures of scene {cfg} variant {variant}")
    ctx.set_scene(sc.desc)
    ctx.build_accel()
    nodes, _, _, info = ctx.read_accel()
    parts = [(int(b[0]), int(b[1]), int(b[3])) for b in info]
    top = max(b + n for b, n, _ in parts)
    parts.append((top, len(nodes) - top, sc.desc.num_instances))
    assert sum(n for _, n, _ in parts) == len(nodes)
    for base, n, prims in parts:
        child, count = nodes[base:base + n, 24:28].astype(np.int64), nodes[base:base + n, 28:32].astype(np.int64)
        empty = child == 0xFFFFFFFF
        inner = ~empty & (count == 0)
        leaf = ~empty & (count > 0)
        assert np.all((child > np.arange(n)[:, None]) | ~inner) and np.all((child < n) | ~inner)
        assert np.array_equal(np.sort(child[inner]), np.arange(1, n))
        assert np.array_equal(np.sort(np.concatenate([np.arange(f, f + c) for f, c in zip(child[leaf], count[leaf])])),
                              np.arange(prims))
