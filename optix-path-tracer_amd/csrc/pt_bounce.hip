// pt_bounce.hip -- launches of the shading kernel, one bounce at a time.
#include "pt_wave.hpp"

namespace pt {

void launch_shade(const DevScene& sc, const DevPaths& P, int in, bool sorted, int out, uint32_t depth,
                  const RenderConsts& rc, int matset, bool count, uint2* spill, uint64_t* stats, int grid,
                  hipStream_t st, const DevScene* scenes, const RenderConsts* rcs, bool batch_env, bool batch_ext) {
  const int src = sorted ? 2 : in;
  const float4* hits = sorted ? P.hit_sorted : P.hit;
  const bool env = (rc.flags & PT_FLAG_ENV_MIS) && sc.num_lights != sc.num_lights_plain;
  const bool cache = (rc.flags & PT_FLAG_RADIANCE_CACHE) != 0;
#define PT_SHADE(MSV, F) \
  launch_shade_v<MSV, F>(sc, P, in, src, hits, out, depth, rc, spill, stats, grid, st, scenes, rcs)
#define PT_SHADE_K(MSV, F, K) \
  launch_shade_v<MSV, F, K>(sc, P, in, src, hits, out, depth, rc, spill, stats, grid, st, scenes, rcs)
  if (scenes && batch_ext) {  // a batch with media, cylinders, moving spheres or the normal shader
    if (batch_env) {
      if (count) PT_SHADE(MS_FULL, SH_MULTI | SH_EXT | SH_ENV | SH_COUNT);
      else PT_SHADE(MS_FULL, SH_MULTI | SH_EXT | SH_ENV);
    } else {
      if (count) PT_SHADE(MS_FULL, SH_MULTI | SH_EXT | SH_COUNT);
      else PT_SHADE(MS_FULL, SH_MULTI | SH_EXT);
    }
  } else if (scenes) {  // a batch of scenes: every material, per-path scene
    if (batch_env) {
      if (count) PT_SHADE(MS_ALL, SH_MULTI | SH_ENV | SH_COUNT);
      else PT_SHADE(MS_ALL, SH_MULTI | SH_ENV);
    } else {
      if (count) PT_SHADE(MS_ALL, SH_MULTI | SH_COUNT);
      else PT_SHADE(MS_ALL, SH_MULTI);
    }
  } else if (sc.wide && (!count || cache)) {  // few scenes: every material and both kinds of lights
    if (matset == MS_FULL || sc.ext_instances != 0) PT_SHADE(MS_FULL, SH_WIDE | SH_EXT | SH_ENV);
    else if (cache) PT_SHADE(MS_ALL, SH_WIDE | SH_CACHE | SH_ENV);
    else PT_SHADE(MS_ALL, SH_WIDE | SH_ENV);
  } else if (matset == MS_FULL || sc.ext_instances != 0) {
    // media or the normal shader (single scenes, no radiance cache)
    if (env) {
      if (count) PT_SHADE(MS_FULL, SH_EXT | SH_ENV | SH_COUNT);
      else PT_SHADE(MS_FULL, SH_EXT | SH_ENV);
    } else {
      if (count) PT_SHADE(MS_FULL, SH_EXT | SH_COUNT);
      else PT_SHADE(MS_FULL, SH_EXT);
    }
  } else if (cache) {  // not asked to count
    if (env) PT_SHADE(MS_ALL, SH_CACHE | SH_ENV);
    else PT_SHADE(MS_ALL, SH_CACHE);
  } else if (env && sc.kinds == 10u) {  // meshes on a ground rect
    if (count) PT_SHADE_K(MS_ALL, SH_ENV | SH_COUNT, 10);
    else PT_SHADE_K(MS_ALL, SH_ENV, 10);
  } else if (env) {
    if (count) PT_SHADE(MS_ALL, SH_ENV | SH_COUNT);
    else PT_SHADE(MS_ALL, SH_ENV);
  } else if (matset == MS_DIFFUSE && (sc.kinds & 8u) == 0) {
    // analytic only (a sphere-free k_shade allocates its registers worse)
    if (count) PT_SHADE_K(MS_DIFFUSE, SH_COUNT, 7);
    else PT_SHADE_K(MS_DIFFUSE, 0, 7);
  } else if (matset == MS_SPHERES && (sc.kinds & 8u) == 0) {
    if (count) PT_SHADE_K(MS_SPHERES, SH_COUNT, 7);
    else PT_SHADE_K(MS_SPHERES, 0, 7);
  } else if (matset == MS_DIFFUSE) {
    if (count) PT_SHADE(MS_DIFFUSE, SH_COUNT);
    else PT_SHADE(MS_DIFFUSE, 0);
  } else if (matset == MS_SPHERES) {
    if (count) PT_SHADE(MS_SPHERES, SH_COUNT);
    else PT_SHADE(MS_SPHERES, 0);
  } else {
    if (count) PT_SHADE(MS_ALL, SH_COUNT);
    else PT_SHADE(MS_ALL, 0);
  }
#undef PT_SHADE_K
#undef PT_SHADE
}

}  // namespace pt
