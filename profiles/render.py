"""One run of a workload for the profiler, from the repository root:

    python3 profiles/render.py meshes | cornell | batch
        one production render, every bounce in launches of its own
    python3 profiles/render.py preview | spheres | next_week
        one render in the default shape (the last bounces in one launch)
    python3 profiles/render.py network
        one training step of the radiance-cache network at 16384 rows and an
        inference over 65537
"""
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "optix-path-tracer_amd"))
import ptamd  # noqa: E402

SCENES = {"meshes": (ptamd.PT_SCENE_MESHES, 0, 0), "cornell": (ptamd.PT_SCENE_CORNELL, 0, 0),
          "preview": (ptamd.PT_SCENE_MESHES, 1920, 1080), "spheres": (ptamd.PT_SCENE_RANDOM_SPHERES, 400, 267),
          "next_week": (ptamd.PT_SCENE_NEXT_WEEK, 301, 203)}
SPP = {"preview": 1, "spheres": 16, "next_week": 16}


def context(scene):
    ctx = ptamd.Context(0)
    ctx.set_scene(scene.desc)
    ctx.build_accel()
    ctx.set_camera(scene.camera)
    return ctx


def main(name):
    if name == "network":
        ctx = ptamd.Context(0)
        ctx.cache_init(1)
        rng = np.random.default_rng(0)
        rows = (rng.random((16384 + 65537, ptamd.PT_CACHE_INPUTS), np.float32).view(np.uint32) >> 16).astype(np.uint16)
        rows[:, 83:] = 0
        ctx.cache_train(rows[:16384], rng.random((16384, 3), np.float32))
        ctx.cache_infer(rows[16384:])
        return "trained and inferred"
    if name == "batch":
        scenes = [ptamd.Scene(ptamd.PT_SCENE_BATCH, 0, 0, k) for k in range(64)]
        params = [s.render_params(flags=s.info.flags | ptamd.PT_FLAG_DIRECT) for s in scenes]
        st = ptamd.render_batch([context(s) for s in scenes], params, [s.info.spp for s in scenes])
    else:
        cfg, w, h = SCENES[name]
        scene = ptamd.Scene(cfg, w, h)
        flags = scene.info.flags | (0 if name in SPP else ptamd.PT_FLAG_DIRECT)
        st = context(scene).render(scene.render_params(flags=flags), 0, SPP.get(name, scene.info.spp))
    return f"{st.gpu_ms:.2f} ms, {st.extend_launches} closest-hit and {st.shade_launches} shading launches"


if __name__ == "__main__":
    print("done", sys.argv[1], main(sys.argv[1]), flush=True)
