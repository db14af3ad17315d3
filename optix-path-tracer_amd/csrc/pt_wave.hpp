// pt_wave.hpp -- the shading kernel of the wavefront integrator and what it
// shares with the other path kernels (wave segments, records, stacks).
#pragma once

#include "pt_kernels.hpp"
#include "pt_shade.hpp"

namespace pt {

// -------------------------------------------------------------- helpers
PTD uint32_t lane_rank(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
// This wave's segment of a path set (layout in pt_layout.hpp).
struct Seg {
  uint32_t stride;  // waves of the grid * row
  uint32_t base;    // w * row
  uint32_t w;       // wave index in the grid
  uint32_t row;     // with fewer than 64 the segment is one row
  PTD uint32_t pos(uint32_t j) const { return (j >> 6) * stride + base + (j & 63u); }
};
PTD Seg my_seg(const DevPaths& P) {
  const uint32_t w = blockIdx.x * WAVES + (threadIdx.x >> 6);
  return Seg{gridDim.x * WAVES * P.row, w * P.row, w, P.row};
}
// positions of the segment below n: the segment count of a dense set
PTD uint32_t dense_count(uint32_t n, const Seg& g) {
  const uint32_t full = n / g.stride, r = n - full * g.stride;
  return full * g.row + (r > g.base ? min(r - g.base, g.row) : 0u);
}
PTD uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
// live paths of this wave's segment of state set `set`
PTD uint32_t seg_count(const DevPaths& P, int set, const Seg& g) {
  return uniform(P.seg[(size_t)set * MAX_WAVES + g.w]);
}
// per-wave statistics row (one writer: lane 0 of the wave)
PTD void stat_add(uint64_t* stats, const Seg& g, int k, uint64_t v) {
  if (v) stats[(size_t)g.w * STAT_WORDS + k] += v;
}

// 24-bit hash of (launch index, frame) choosing radiance-cache training
// paths; independent of the path's own random sequence
PTD uint32_t train_hash(uint32_t pix, uint32_t frame) {
  uint32_t h = pix * 0x9E3779B1u ^ (frame + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  h *= 0x297A2D39u;
  h ^= h >> 15;
  return h >> 8;
}

// Radiance-cache input features, 96 BF16 (83 used, the rest zero):
//   [0, 72)   sin, cos (2^f pi p), f = 0..11, per axis of the position p
//             normalised to the scene box (angle doubling from pi p)
//   [72, 74)  view direction Wo as (theta / pi, phi / 2 pi + 1/2), theta from +Y
//   [74, 76)  shading normal, same mapping
//   76        roughness, [77, 80) diffuse albedo, [80, 83) specular albedo
PTD uint32_t bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return u >> 16;
}
struct FeatWriter {
  uint4* dst;
  float buf[8];
  int n = 0, k = 0;
  PTD void put(float v) {
    buf[n++] = v;
    if (n == 8) {
      dst[k++] = make_uint4(bf16_bits(buf[0]) | (bf16_bits(buf[1]) << 16), bf16_bits(buf[2]) | (bf16_bits(buf[3]) << 16),
                            bf16_bits(buf[4]) | (bf16_bits(buf[5]) << 16), bf16_bits(buf[6]) | (bf16_bits(buf[7]) << 16));
      n = 0;
    }
  }
};
PTD void sph_dir(v3 w, float& a, float& b) {
  a = pacos(fminf(fmaxf(w.y, -1.f), 1.f)) * (1.f / PI_F);
  b = patan2(w.z, w.x) * (0.5f / PI_F) + 0.5f;
}
__device__ __attribute__((noinline)) void write_features(uint4* dst, const CacheConsts& cc, v3 P, v3 Wo, v3 N,
                                                         const Surface& f) {
  FeatWriter fw{dst};
  const float pp[3] = {(P.x - cc.lo[0]) * cc.inv_ext[0], (P.y - cc.lo[1]) * cc.inv_ext[1],
                       (P.z - cc.lo[2]) * cc.inv_ext[2]};
  for (int a = 0; a < 3; a++) {
    float sn = psin(PI_F * pp[a]), cs = pcos(PI_F * pp[a]);
    for (int q = 0; q < 12; q++) {
      fw.put(sn);
      fw.put(cs);
      float s2 = 2.f * sn * cs, c2 = cs * cs - sn * sn;
      sn = s2;
      cs = c2;
    }
  }
  float a, b;
  sph_dir(normalize(Wo), a, b);
  fw.put(a);
  fw.put(b);
  sph_dir(normalize(N), a, b);
  fw.put(a);
  fw.put(b);
  float rough = 1.f;
  v3 rd = mk3(0.f), rs = mk3(0.f);
  switch (f.type) {
    case PT_MAT_LAMBERTIAN:
    case PT_MAT_OREN_NAYAR: rd = f.c0; break;
    case PT_MAT_METAL: rough = f.p0; rs = f.c0; break;
    case PT_MAT_DIELECTRIC: rough = 0.f; rs = mk3(1.f); break;
    case PT_MAT_ASHIKHMIN_SHIRLEY: rough = 1.f / sqrtf(1.f + 0.5f * (f.p0 + f.p1)); rd = f.c0; rs = f.c1; break;
    case PT_MAT_TORRANCE_SPARROW: rough = sqrtf(f.p0); rs = f.c0; break;
    default: break;
  }
  fw.put(rough);
  fw.put(rd.x);
  fw.put(rd.y);
  fw.put(rd.z);
  fw.put(rs.x);
  fw.put(rs.y);
  fw.put(rs.z);
  while (fw.k < 12) fw.put(0.f);
}

template <int NL = STK_LDS>
PTD StackT<NL> make_stack(uint2* s_stk, uint2* spill, uint32_t* overflow) {
  StackT<NL> st;
  st.lds = s_stk + threadIdx.x;
  st.spill = spill + (size_t)(blockIdx.x * BLOCK + threadIdx.x) * STK_TOTAL;
  st.sp = 0;
  st.overflow = overflow;
  return st;
}

// Throughput (w: pdf of the previous bounce) and radiance (w: path signature,
// the FNV-1a offset basis) of every path before its first bounce.  The first
// shading pass (depth 0) takes them from here, so the path start does not
// store them: state set 0 holds only o and d until depth 1 rewrites it
// (max_depth >= 1; the material sort copies the unset T and L of depth 0,
// which nothing reads).
PTD float4 path_T0() { return make_float4(1.f, 1.f, 1.f, 1.f); }
PTD float4 path_L0() { return make_float4(0.f, 0.f, 0.f, __uint_as_float(0x811C9DC5u)); }

// Scatter of the materials that do not sample lights plus the continuation
// sample of Lambertian / Oren-Nayar, then Russian roulette (raygen.cu:96-118).
// Returns false when the path ended (result written).
template <int MS>
PTD bool scatter_and_roulette(const Surface& f, v3 Wo, v3 N, uint32_t& seed, uint32_t& sig, v3& T, v3 L, v3& dir,
                              uint32_t& flags, float& prev_pdf, uint32_t depth, const RenderConsts& rc,
                              float4& result) {
  bool spec = false;
  if ((has_mat<MS>(PT_MAT_LAMBERTIAN) || has_mat<MS>(PT_MAT_OREN_NAYAR)) &&
      (f.type == PT_MAT_LAMBERTIAN || f.type == PT_MAT_OREN_NAYAR)) {
    // lambertian.cu:62-72, oren_nayar.cu:59-69
    v3 Wi = brdf_sample<MS>(f, Wo, N, seed);
    float pdf = 1.f;
    v3 att = brdf_eval<MS>(f, Wo, Wi, N, pdf);
    dir = Wi;
    T = T * clamp3(att / pdf, 0.f, 1.f);
    prev_pdf = pdf;
  } else if (has_mat<MS>(PT_MAT_METAL) && f.type == PT_MAT_METAL) {  // metal.cu:38-56
    v3 refl = reflect(-Wo, N);
    dir = refl + f.p0 * random_in_unit_sphere(seed);
    T = T * f.c0;
    spec = true;
  } else if (has_mat<MS>(PT_MAT_DIELECTRIC) && f.type == PT_MAT_DIELECTRIC) {  // dielectric.cu:46-96
    float ior = f.p0;
    v3 W = -Wo;
    v3 Nd = N;
    float ni_over_nt;
    float cosine = dot(W, Nd);
    if (cosine > 0.f) {
      Nd = -Nd;
      ni_over_nt = ior;
      cosine = ior * cosine / length(W);
    } else {
      ni_over_nt = 1.f / ior;
      cosine = -cosine / length(W);
    }
    v3 refracted = mk3(0.f);
    float reflect_prob;
    if (Refract(W, Nd, ni_over_nt, refracted)) reflect_prob = schlick(cosine, ior);
    else reflect_prob = 1.f;
    bool refl = rnd(seed) < reflect_prob;
    sig = sig_mix(sig, refl ? 0x11111111u : 0x22222222u);
    dir = refl ? reflect(W, Nd) : normalize(refracted);
    T = T * f.c0;
    spec = true;
  } else if (has_mat<MS>(PT_MAT_ASHIKHMIN_SHIRLEY) && f.type == PT_MAT_ASHIKHMIN_SHIRLEY) {
    // ashikhmin_shirley.cu:48-68
    v3 Wi = brdf_sample<MS>(f, Wo, N, seed);
    float pdf = 1.f;
    v3 att = brdf_eval<MS>(f, Wo, Wi, N, pdf);
    dir = Wi;
    T = T * clamp3(att, 0.f, 1.f);
    spec = true;
  } else if (has_mat<MS>(PT_MAT_ISOTROPIC) && f.type == PT_MAT_ISOTROPIC) {  // isotropic.cu:42-50
    v3 Wi = brdf_sample<MS>(f, Wo, N, seed);
    float pdf = 1.f;
    v3 att = brdf_eval<MS>(f, Wo, Wi, N, pdf);
    dir = Wi;
    T = T * (att / pdf);
    prev_pdf = pdf;
  } else if (has_mat<MS>(PT_MAT_TORRANCE_SPARROW)) {  // Torrance-Sparrow, torrance_sparrow.cu:39-59
    v3 Wi = brdf_sample<MS>(f, Wo, N, seed);
    float pdf = 1.f;
    v3 att = brdf_eval<MS>(f, Wo, Wi, N, pdf);
    dir = Wi;
    T = T * clamp3(att / pdf, 0.f, 1.f);
    spec = true;
  }
  flags = spec ? 1u : 0u;
  if (rc.russian) {
    float prob = max_component(T);
    if (depth >= rc.rr_min_depth) {
      bool term = rnd(seed) >= prob;
      sig = sig_mix(sig, term ? 0x44444444u : 0x55555555u);
      if (term) {
        v3 r = L + T;
        result = make_float4(r.x, r.y, r.z, __uint_as_float(depth + 1));
        return false;
      }
      T = T * (1.f / prob);
    }
  }
  return true;
}

// Closest-hit / miss programs of every live path for one bounce: hit record,
// Direct_Light with its shadow ray traced here (light_sample.cuh:35-103;
// lit iff the closest hit in (1e-3, inf) is a diffuse light with
// dot(N, Wi) > 0, or nothing is hit), the emitter rules, the continuation
// sample and Russian roulette.  Surviving paths are appended, wave by wave,
// to state set `out`; finished paths write their slot's result.
// FEAT: SH_COUNT counts the shadow rays' traversal, SH_CACHE records
// radiance-cache training vertices and queries, SH_ENV samples environment
// lights, SH_EXT traces shadow rays through volumes, SH_WIDE takes 64-bit node
// addresses (one scene of 4 GB of nodes or more); each is compiled only into
// the variants that use it.
//
// SH_TAIL (depth0 >= 1 and beyond the cache's query depth, in == src): the launch runs every bounce that is
// left.  A wave traces the closest hit of its 64 paths itself, shades them,
// and goes on with its segment's survivors (the two state sets in turn)
// until none is left, so the waves wait neither for each other nor for a
// launch.  Once a bounce has few paths per wave, its own launches last as
// long as the longest ray of the whole batch (about 0.6 us per traversal
// step: 250 us in the mesh scene, 40 us in the sphere scene) plus 35 us of
// material sort, whatever the number of paths; a wave's own chain of rays
// is shorter than the sum of the batch's longest ones.  The paths' results
// do not depend on the order they are traced in: images are the same bit
// for bit.  Against a launch per kernel and bounce, the kernels otherwise as
// they were then: 64x64 Cornell tile 526 -> 339 us, random spheres 4.29 ->
// 1.9 ms, next-week scene 10.5 -> 4.1 ms, one 1080p frame of the mesh scene
// 6.0 -> 4.6 ms (270 us, 1.5, 3.5 and 3.4 ms with the traversal and the
// spread of small batches of today; 7.6 to 13 lanes are busy per instruction).
constexpr int SH_COUNT = 1, SH_CACHE = 2, SH_ENV = 4, SH_MULTI = 8, SH_EXT = 16, SH_TAIL = 32, SH_WIDE = 64;
template <int MS, int FEAT, int KINDS = KIND_ALL>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_shade(
    DevScene sc0, DevPaths P, int in, int src, const float4* __restrict__ hits, int out, uint32_t depth0,
    RenderConsts rc0, uint2* spill, uint64_t* stats, const DevScene* __restrict__ scenes,
    const RenderConsts* __restrict__ rcs) {
  constexpr bool MULTI = (FEAT & SH_MULTI) != 0;
  constexpr bool EXT = (FEAT & SH_EXT) != 0;
  constexpr bool WIDE = (FEAT & (SH_MULTI | SH_WIDE)) != 0;
  __shared__ uint2 s_stk[STK_LDS_SHADE * BLOCK];
  // each lane's T, L, normal and view direction wait here while its shadow
  // ray is traced: fewer registers live across the traversal (fewer scratch
  // spills; with the stack, 36 KB per block keeps 4 blocks of 4 waves per CU)
  __shared__ float s_keep[12 * BLOCK];
  StackT<STK_LDS_SHADE> st = make_stack<STK_LDS_SHADE>(s_stk, spill, P.counters + CTR_STACK_OVERFLOW);
  const Seg g = my_seg(P);
  uint32_t depth = depth0;
  uint32_t n = seg_count(P, src, g);
  PathState S = P.st[src], D = P.st[out];
  uint32_t survivors = 0;  // wave-uniform: paths written to this wave's segment of `out`
  constexpr bool COUNT = (FEAT & SH_COUNT) != 0;
  constexpr bool TAIL = (FEAT & SH_TAIL) != 0;
  uint32_t ext_rays = 0;  // TAIL: closest-hit queries of this wave
  const bool cache_on = !MULTI && (FEAT & SH_CACHE) && (rc0.flags & PT_FLAG_RADIANCE_CACHE) != 0;
  TraceCounts tc{0, 0, 0};
  uint32_t shadow_rays = 0, exhausted = 0;
  // radiance-cache records of this wave (wave-uniform running counts):
  // training vertices continue the batch's count, queries start at zero
  uint32_t tcount = 0, qcount = 0, tcap = 0;
  if (cache_on) {
    tcount = uniform(P.tseg[g.w]);
    tcap = dense_count(P.t_cap, g);
  }
  do {  // TAIL: one trip per bounce, else once
    if (TAIL) {
      ext_rays += n;
      survivors = 0;
    }
    for (uint32_t j0 = 0; j0 < n; j0 += 64) {
      const uint32_t i = g.pos(j0 + __lane_id());
      bool alive = false, did_rec = false, did_ask = false;
      float4 no = make_float4(0.f, 0.f, 0.f, 0.f), nd = no, nT = no, nL = no;
      if (j0 + __lane_id() < n) {
        float4 hit;
        float4 o4 = S.o[i], d4 = S.d[i];
        if (TAIL) {
          const DevScene& tsc = MULTI ? scenes[__float_as_uint(o4.w) >> 24] : sc0;
          const float ttm = (EXT && tsc.mov_instances) ? P.ptime[__float_as_uint(d4.w) & SLOT_MASK] : 0.f;
          const HitOut th = trace_closest<false, EXT, KINDS, false, WIDE>(tsc, mk3(o4), mk3(d4), 1e-3f, FINF, st, tc,
                                                             __float_as_uint(o4.w), ttm);
          hit = make_float4(th.t, __int_as_float(th.pos), __int_as_float(th.prim), 0.f);
        } else {
          hit = hits[i];
        }
        const float4 t4 = depth == 0 ? path_T0() : S.T[i], l4 = depth == 0 ? path_L0() : S.L[i];
        v3 d = mk3(d4), T = mk3(t4), L = mk3(l4);
        uint32_t seed = __float_as_uint(o4.w), dw = __float_as_uint(d4.w);
        // a batch of scenes keeps the path's scene in the RNG state's top
        // byte (the 24-bit outputs never depend on it)
        const uint32_t sid = MULTI ? (seed >> 24) : 0u;
        const DevScene& sc = MULTI ? scenes[sid] : sc0;
        const RenderConsts& rc = MULTI ? rcs[sid] : rc0;
        // light table: environment lights take part only with PT_FLAG_ENV_MIS
        const bool env_mis = (FEAT & SH_ENV) && (rc.flags & PT_FLAG_ENV_MIS) != 0;
        const DevLight* lights = env_mis ? sc.lights : sc.lights_plain;
        const int nl = env_mis ? sc.num_lights : sc.num_lights_plain;
        const bool env_light = env_mis && sc.env_total != 0 && sc.num_lights != sc.num_lights_plain;
        // dw keeps slot | TRAIN_BIT | SPEC_BIT; fields are taken where used
        uint32_t flags = dw >> 31, sig = __float_as_uint(l4.w);
        float prev_pdf = t4.w;
        int pos = __float_as_int(hit.y), prim = __float_as_int(hit.z);
        sig = sig_mix(sig, pos >= 0 ? (((uint32_t)inst_at(sc, pos) << 20) ^ (uint32_t)prim) : 0xFFFFFFFFu);
        float4 res = make_float4(0.f, 0.f, 0.f, 0.f);
        if (pos < 0) {
          if (env_mis && sc.miss.type == PT_MISS_HDR) {
            // unclamped environment radiance, MIS-weighted against the light
            // sample of the previous (diffuse) bounce
            v3 Le = env_radiance(sc, d);
            float w = 1.f;
            if (env_light && depth > 0 && !(flags & 1u)) w = power_heuristic(prev_pdf, env_pdf(sc, d));
            T = T * (Le * w);
            v3 r = L + T;
            res = make_float4(r.x, r.y, r.z, __uint_as_float(depth + 1));
          } else {
            // miss programs (miss.cu), then color() returns L + clamp(T) (raygen.cu:81-82)
            T = T * miss_color(sc, d);
            v3 r = L + clamp3(T, 0.f, 1.f);
            res = make_float4(r.x, r.y, r.z, __uint_as_float(depth + 1));
          }
        } else {
          int mat = hit_material(sc, pos, prim);
          const DevMaterial& M = gp(sc.mats)[mat];
          bool need_uv = tex_needs_uv(sc, M.tex0) || (M.type == PT_MAT_ASHIKHMIN_SHIRLEY && tex_needs_uv(sc, M.tex1));
          const float tm = (EXT && sc.mov_instances) ? P.ptime[dw & SLOT_MASK] : 0.f;
          HitRec r = hit_record<KINDS, EXT>(sc, pos, prim, hit.x, mk3(o4), d, need_uv, tm);
          Surface f = make_surface(sc, r);
          bool is_light = has_mat<MS>(PT_MAT_DIFFUSE_LIGHT) && f.type == PT_MAT_DIFFUSE_LIGHT;
          // the isotropic medium samples lights without the hemisphere test of
          // light_sample.cuh:60 and :71 (its +X normal is not a surface's)
          const bool iso = has_mat<MS>(PT_MAT_ISOTROPIC) && f.type == PT_MAT_ISOTROPIC;
          bool nee = ((has_mat<MS>(PT_MAT_LAMBERTIAN) || has_mat<MS>(PT_MAT_OREN_NAYAR)) &&
                      (f.type == PT_MAT_LAMBERTIAN || f.type == PT_MAT_OREN_NAYAR)) || is_light || iso;
          bool queried = false;
          if (cache_on) {
            // training paths record every vertex (radiance so far, throughput);
            // other paths end at the query depth with a cache lookup
            // (every lane with rec or ask is active here, so the ballots rank
            // exactly the lanes the converged counts below add up)
            const bool rec = (dw & TRAIN_BIT) != 0;
            const bool ask = !rec && depth == rc.cache.query_depth;
            const uint32_t tj = tcount + lane_rank(__ballot(rec));
            const uint32_t qj = qcount + lane_rank(__ballot(ask));
            did_rec = rec;
            did_ask = ask;
            if (rec && tj < tcap) {
              const uint32_t k = g.pos(tj);
              write_features(P.t_feat + (size_t)k * 12, rc.cache, r.P, r.Wo, r.N, f);
              P.t_L[k] = make_float4(L.x, L.y, L.z, __uint_as_float(dw & SLOT_MASK));
              P.t_T[k] = make_float4(T.x, T.y, T.z, 0.f);
            }
            if (ask) {
              // queries never outnumber the wave's inputs: the position exists
              queried = true;
              const uint32_t k = g.pos(qj);
              write_features(P.q_feat + (size_t)k * 12, rc.cache, r.P, r.Wo, r.N, f);
              P.q_meta[k] = make_float4(T.x, T.y, T.z, __uint_as_float(dw & SLOT_MASK));
              res = make_float4(L.x, L.y, L.z, __uint_as_float(depth + 1));
              nee = false;
            }
          }
          if (nee) {
            v3 direct = mk3(0.f);
            if (nl > 0) {
              int index = ((int)(rnd(seed) * nl)) % nl;
              if (!(is_light && nl == 1)) {
                const DevLight& Lt = gp(lights)[index];
                const bool env = (FEAT & SH_ENV) && Lt.type == PT_LIGHT_ENV;
                v3 Wi = env ? env_sample(sc, seed) : light_sample(Lt, r.P, seed);
                float lightPDF = env ? env_pdf(sc, Wi) : light_pdf(Lt, r.P, Wi);
                if (!iso && dot(Wi, r.N) < 0.f) {
                  sig = sig_mix(sig, 0x33333333u);
                } else {
                  shadow_rays++;
                  const uint32_t kt = threadIdx.x;
                  auto keep = [&](int k, v3 v) {
                    s_keep[k * BLOCK + kt] = v.x;
                    s_keep[(k + 1) * BLOCK + kt] = v.y;
                    s_keep[(k + 2) * BLOCK + kt] = v.z;
                  };
                  auto kept = [&](int k) {
                    return mk3(s_keep[k * BLOCK + kt], s_keep[(k + 1) * BLOCK + kt], s_keep[(k + 2) * BLOCK + kt]);
                  };
                  keep(0, T);
                  keep(3, L);
                  keep(6, r.N);
                  keep(9, r.Wo);
                  // an environment sample is lit iff its shadow ray hits
                  // nothing (any hit occludes): the first hit found decides it
                  HitOut sh = trace_closest<COUNT, EXT, KINDS, true, WIDE>(sc, r.P, Wi, 1e-3f, FINF, st, tc, seed, tm, env);
                  T = kept(0);
                  L = kept(3);
                  r.N = kept(6);
                  r.Wo = kept(9);
                  const v3 emission = env ? env_radiance(sc, Wi) : light_emission(Lt);
                  bool occluded = false;
                  if (sh.pos >= 0)
                    occluded = env || !(gp(sc.mats)[hit_material(sc, sh.pos, sh.prim)].type == PT_MAT_DIFFUSE_LIGHT &&
                                        (iso || dot(r.N, Wi) > 0.f));
                  sig = sig_mix(sig, occluded ? 0xA5A5A5A5u : 0x5A5A5A5Au);
                  if (!occluded) {
                    if (lightPDF != 0.f && !isNull(emission)) {
                      float matPDF = 1.f;
                      v3 mv = brdf_eval<MS>(f, r.Wo, Wi, r.N, matPDF);
                      if (matPDF != 0.f && !isNull(mv)) {
                        float w = power_heuristic(lightPDF, matPDF);
                        direct = direct + mv * emission * w / lightPDF;
                      }
                    }
                    if (!env) {
                      v3 Wb = brdf_sample<MS>(f, r.Wo, r.N, seed);
                      float matPDF = 1.f;
                      v3 mv = brdf_eval<MS>(f, r.Wo, Wb, r.N, matPDF);
                      if (matPDF != 0.f && !isNull(mv)) {
                        float lp = light_pdf(Lt, r.P, Wb);
                        if (lp != 0.f && !isNull(emission)) {
                          float w = power_heuristic(matPDF, lp);
                          direct = direct + mv * emission * w / matPDF;
                        }
                      }
                    }
                  }
                }
              }
            }
            L = L + T * direct;
          }
          if (queried) {
            // result = L now; the cache adds T * radiance after inference
          } else if (has_mat<MS>(PT_MAT_NORMAL) && f.type == PT_MAT_NORMAL) {
            // normal_shader.cu:22-34: the radiance becomes 0.5 N + 0.5 and the
            // path is cancelled (color() returns it)
            v3 nn = f.p0 != 0.f ? r.N : geometric_normal(sc, pos, prim, r.N);
            v3 c = nn * 0.5f + mk3(0.5f);
            res = make_float4(c.x, c.y, c.z, __uint_as_float(depth + 1));
          } else if (is_light) {
            // diffuse_light.cu:43-47 and raygen.cu:85-90
            if (dot(r.N, r.Wo) < 0.f) T = T * f.c0;
            if (depth == 0 || (flags & 1u)) L = L + T;
            res = make_float4(L.x, L.y, L.z, __uint_as_float(depth + 1));
          } else {
            v3 ndir;
            alive = scatter_and_roulette<MS>(f, r.Wo, r.N, seed, sig, T, L, ndir, flags, prev_pdf, depth, rc, res);
            if (alive) {
              no = make_float4(r.P.x, r.P.y, r.P.z, __uint_as_float(MULTI ? ((seed & 0xFFFFFFu) | (sid << 24)) : seed));
              nd = make_float4(ndir.x, ndir.y, ndir.z, __uint_as_float((dw & ~SPEC_BIT) | (flags << 31)));
              nT = make_float4(T.x, T.y, T.z, prev_pdf);
              nL = make_float4(L.x, L.y, L.z, __uint_as_float(sig));
            }
          }
        }
        if ((MULTI || TAIL) && alive && depth + 1 >= rc.max_depth) {
          // the last bounce of this path's scene: it ends like the paths that
          // outlive a single scene's loop (k_exhausted), result left as the
          // path start set it
          alive = false;
          exhausted++;
          P.sig_final[dw & SLOT_MASK] = sig;
        } else if (!alive) {
          P.result[dw & SLOT_MASK] = res;
          P.sig_final[dw & SLOT_MASK] = sig;
        }
      }
      // compaction of the survivors into this wave's segment of set `out`
      // (never more than the wave's inputs, so every position exists)
      const uint64_t mask = __ballot(alive);
      if (alive) {
        const uint32_t k = g.pos(survivors + lane_rank(mask));
        D.o[k] = no;
        D.d[k] = nd;
        D.T[k] = nT;
        D.L[k] = nL;
      }
      survivors += (uint32_t)__popcll(mask);
      if (cache_on) {
        tcount = min(tcount + (uint32_t)__popcll(__ballot(did_rec)), tcap);
        qcount += (uint32_t)__popcll(__ballot(did_ask));
      }
    }
    if (TAIL) {
      // the survivors of this bounce are the wave's paths of the next one; the
      // fence makes what other lanes stored visible to the next loads
      __threadfence_block();
      n = survivors;
      const PathState X = S;
      S = D;
      D = X;
      depth++;
    }
  } while (TAIL && n != 0);
  uint32_t a = tc.nodes, b = tc.prims, c = tc.insts;
  for (int off = 32; off > 0; off >>= 1) {
    shadow_rays += __shfl_down(shadow_rays, off);
    if (MULTI || TAIL) exhausted += __shfl_down(exhausted, off);
    if (COUNT) {
      a += __shfl_down(a, off);
      b += __shfl_down(b, off);
      c += __shfl_down(c, off);
    }
  }
  if (__lane_id() == 0) {
    if (!TAIL) P.seg[(size_t)out * MAX_WAVES + g.w] = survivors;
    if (TAIL) stat_add(stats, g, STAT_EXT, ext_rays);
    if (cache_on) {
      P.tseg[g.w] = tcount;
      if (depth == rc0.cache.query_depth) P.qseg[g.w] = qcount;
    }
    stat_add(stats, g, STAT_SHADOW, shadow_rays);
    if (MULTI || TAIL) stat_add(stats, g, STAT_EXHAUSTED, exhausted);
    if (COUNT) {
      stat_add(stats, g, STAT_SH_NODES, a);
      stat_add(stats, g, STAT_SH_PRIMS, b);
      stat_add(stats, g, STAT_SH_INSTS, c);
    }
  }
}

template <int MS, int FEAT, int KINDS = KIND_ALL>
static inline void launch_shade_v(const DevScene& sc, const DevPaths& P, int in, int src, const float4* hits, int out,
                           uint32_t depth, const RenderConsts& rc, uint2* spill, uint64_t* stats, int grid,
                           hipStream_t st, const DevScene* scenes, const RenderConsts* rcs) {
  hipLaunchKernelGGL((k_shade<MS, FEAT, KINDS>), dim3(grid), dim3(BLOCK), 0, st, sc, P, in, src, hits, out, depth, rc, spill,
                     stats, scenes, rcs);
}

}  // namespace pt
