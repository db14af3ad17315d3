// pt_tail.hip -- launches of the shading kernel that run every bounce left.
#include "pt_wave.hpp"

namespace pt {

void launch_tail(const DevScene& sc, const DevPaths& P, int in, int out, uint32_t depth, const RenderConsts& rc,
                 int matset, uint2* spill, uint64_t* stats, int grid, hipStream_t st, const DevScene* scenes,
                 const RenderConsts* rcs, bool batch_env, bool batch_ext) {
  const bool env = (rc.flags & PT_FLAG_ENV_MIS) && sc.num_lights != sc.num_lights_plain;
#define PT_TAIL(MSV, F, K) \
  launch_shade_v<MSV, (F) | SH_TAIL, K>(sc, P, in, in, nullptr, out, depth, rc, spill, stats, grid, st, scenes, rcs)
  if (scenes && batch_ext) {
    if (batch_env) PT_TAIL(MS_FULL, SH_MULTI | SH_EXT | SH_ENV, KIND_ALL);
    else PT_TAIL(MS_FULL, SH_MULTI | SH_EXT, KIND_ALL);
  } else if (scenes) {
    if (batch_env) PT_TAIL(MS_ALL, SH_MULTI | SH_ENV, KIND_ALL);
    else PT_TAIL(MS_ALL, SH_MULTI, KIND_ALL);
  } else if (sc.wide) {
    if (matset == MS_FULL || sc.ext_instances != 0) PT_TAIL(MS_FULL, SH_WIDE | SH_EXT | SH_ENV, KIND_ALL);
    else if (rc.flags & PT_FLAG_RADIANCE_CACHE) PT_TAIL(MS_ALL, SH_WIDE | SH_CACHE | SH_ENV, KIND_ALL);
    else PT_TAIL(MS_ALL, SH_WIDE | SH_ENV, KIND_ALL);
  } else if (matset == MS_FULL || sc.ext_instances != 0) {
    if (env) PT_TAIL(MS_FULL, SH_EXT | SH_ENV, KIND_ALL);
    else PT_TAIL(MS_FULL, SH_EXT, KIND_ALL);
  } else if (rc.flags & PT_FLAG_RADIANCE_CACHE) {
    if (env) PT_TAIL(MS_ALL, SH_CACHE | SH_ENV, KIND_ALL);
    else PT_TAIL(MS_ALL, SH_CACHE, KIND_ALL);
  } else if (env && sc.kinds == 10u) {
    PT_TAIL(MS_ALL, SH_ENV, 10);
  } else if (env) {
    PT_TAIL(MS_ALL, SH_ENV, KIND_ALL);
  } else if (matset == MS_DIFFUSE && (sc.kinds & 8u) == 0) {
    PT_TAIL(MS_DIFFUSE, 0, 7);
  } else if (matset == MS_SPHERES && (sc.kinds & 8u) == 0) {
    PT_TAIL(MS_SPHERES, 0, 7);
  } else {
    PT_TAIL(MS_ALL, 0, KIND_ALL);
  }
#undef PT_TAIL
}

}  // namespace pt
