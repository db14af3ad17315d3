// pt_trace.hpp -- two-level BVH4 closest-hit traversal (replaces OptiX's
// rtTrace: programs/raygen.cu:77, programs/materials/light_sample.cuh:69).
//
// One ray per lane.  The traversal stack keeps its top entries in LDS (one
// column per lane, bank-conflict free; how many is the kernel's choice) and
// spills deeper entries to a per-thread slice of HBM.  Children are visited
// nearest first by entry distance (node_fast's has a margin); popped entries
// farther than the current hit are skipped.
// Candidates win on smaller t, ties on the smaller (instance, primitive) key,
// so the result does not depend on visit order.
#pragma once

#include "pt_device.hpp"

namespace pt {

template <int NL>
struct StackT {
  uint2* lds;    // LDS column (reference, entry distance), stride BLOCK
  uint2* spill;  // this thread's HBM slice (STK_TOTAL entries)
  int sp;
  uint32_t* overflow;
  PTD void put(int pos, uint32_t r, float t) {
    if (pos < NL) {
      lds[pos * BLOCK] = make_uint2(r, __float_as_uint(t));
    } else if (pos < STK_TOTAL) {
      spill[pos - NL] = make_uint2(r, __float_as_uint(t));
    } else {
      atomicAdd(overflow, 1u);
    }
  }
  PTD void pop(uint32_t& r, float& t) {
    sp--;
    uint2 e = make_uint2(EMPTY_REF, __float_as_uint(FINF));
    if (sp < NL) e = lds[sp * BLOCK];
    else if (sp < STK_TOTAL) e = spill[sp - NL];
    r = e.x;
    t = __uint_as_float(e.y);
  }
  // three entries fit the LDS part in every lane
  PTD bool room() const { return __ballot(sp > NL - 3) == 0; }
  PTD void push_lds(uint32_t r, float t) {
    lds[sp * BLOCK] = make_uint2(r, __float_as_uint(t));
    sp++;
  }
};
using Stack = StackT<STK_LDS>;

PTD float4 as_f4(uint4 u) {
  return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
}

struct HitOut {
  float t;
  int prim;  // original primitive index (-1: miss)
  int pos;   // instance position in top-level order (-1: miss)
};
// original instance id of the instance at top-level position pos
PTD int inst_at(const DevScene& sc, int pos) { return (int)gp(sc.insts)[(size_t)pos * 8 + 3].w; }

struct TraceCounts {
  uint32_t nodes, prims, insts;
};

// entry distance of one child slot or +inf
PTD float slab_test(float lox, float hix, float loy, float hiy, float loz, float hiz, v3 o, v3 inv, float tmin,
                    float tmax) {
  float t0x = (lox - o.x) * inv.x, t1x = (hix - o.x) * inv.x;
  float t0y = (loy - o.y) * inv.y, t1y = (hiy - o.y) * inv.y;
  float t0z = (loz - o.z) * inv.z, t1z = (hiz - o.z) * inv.z;
  float tn = fmaxf(fmaxf(fminf(t0x, t1x), fminf(t0y, t1y)), fmaxf(fminf(t0z, t1z), tmin));
  float tf = fminf(fminf(fmaxf(t0x, t1x), fmaxf(t0y, t1y)), fminf(fmaxf(t0z, t1z), tmax));
  return (tn <= tf * SLAB_FAR_SCALE) ? tn : FINF;
}

// EXT: the scene holds instances of the extended kinds (volumes,
// cylinders, moving spheres); volume free flights are drawn from `vseed`
// (the ray's RNG state) and the volume and instance ids, moving spheres are
// placed at `time`.
// KINDS: bit k set when instances of PT_GEOM kind k (spheres, rects,
// boxes, meshes) may occur; the tests of the other kinds (and the
// triangle test's per-instance ray setup) are compiled out.
constexpr int KIND_ALL = 15;
// Every loop here ends because the structure is a tree: the builder gives a
// child node a larger index than its parent and one parent only, so a descent
// is no longer than the levels and every entry pushed is popped once.
// TRIPS_MAX also ends a wave whose memory was overwritten: it bounds the calls
// of step() for a wave's lock-step rays, or since rays were last handed to its
// idle lanes; past it the rays in hand end with what they have found.  (The
// nodes that one step() visits in scenes with meshes are not counted: a count
// in that loop took rays_device 563 -> 588 us and the mesh and next-week stills
// 1 to 2 % more.)
constexpr uint32_t TRIPS_MAX = 1u << 22;
// The traversal of one ray as a resumable state: begin() sets it up, each
// step() does one trip of the loop (see there) and returns false once the ray
// is done (h then holds the result).  trace_closest runs the steps back to back;
// kernels that refill lanes with new rays step several rays at once.
//
// ANY && any_hit: the ray ends at the first candidate accepted in
// (tmin, tmax) instead of the closest (occlusion queries whose answer is
// only whether anything is hit: a miss is a miss either way, and a hit is
// reported as one).  ANY is a template switch so that the closest-hit
// kernels carry no trace of the early exit (a runtime-false flag still
// changes their traversal loop's code and costs them about a tenth of
// their time).
//
// QUERY: a caller's rays, whose directions may have any length (see
// fast_setup).
template <bool COUNT, bool EXT = false, int KINDS = KIND_ALL, bool ANY = false, bool WIDE = false, bool QUERY = false>
struct Tracer {
  static constexpr bool SPH = (KINDS & 1) != 0, RECT = (KINDS & 2) != 0, BOX = (KINDS & 4) != 0,
                        MESH = (KINDS & 8) != 0;
  // FAST (kernels that do not count): the node test of node_fast
  static constexpr bool FAST = !COUNT;
  // rect and box tests (and the exact slab test) take the IEEE reciprocal
  // direction: kept per instance, or, next to meshes (no registers to spare),
  // formed by each test
  static constexpr bool KEEP_INV = COUNT || ((RECT || BOX) && !MESH);
  HitOut h;
  v3 o, d, ro, rd, rinv;
  // FAST: bounded reciprocal direction; -o * inv moved outward for near and
  // far planes; byte offsets of the near planes in a node
  v3 finv, nb, fb;
  uint32_t sx, sy, sz;
  float scale;  // QUERY: node distances are t * scale
  float tmin, time;
  uint32_t vseed;
  TriRay tr;
  int cur;      // instance slot in top-level order, -1 = top level
  int base_sp;  // stack depth when the instance was entered
  uint32_t node_base, prim_base, kind;
  // WIDE: the address of node node_base instead (a batch's kernels would
  // fetch the node array's address from the scene's table entry at each node)
  uint64_t node_ptr;
  bool moved;   // the instance in hand has a transform: ro, rd are its own
  // the entry in hand: the top-level root first; the nearest child of each
  // node and an instance's root are taken directly instead of through the
  // stack, which visits the same nodes in the same order
  uint32_t ref;
  bool have, any_hit;

  // a candidate of the instance in hand as far as the hit: the smaller
  // (instance, primitive) wins
  PTD bool wins_tie(const DevScene& sc, int orig) const {
    const int a = inst_at(sc, cur), b = inst_at(sc, h.pos);
    return a < b || (a == b && orig < h.prim);
  }
  PTD v3 exact_inv() const {
    return KEEP_INV ? rinv : mk3(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
  }

  // the watertight test of one triangle record and, when it is nearer (or
  // as near with the smaller key), its acceptance; true when an any-hit
  // query ends here
  PTD bool offer_tri(const DevScene& sc, float4 a, float4 b, float4 c, TraceCounts& cnt) {
    if (COUNT) cnt.prims++;
    float t = FINF, b1, b2;
    if (!tri_test(tr, ro, mk3(a), mk3(b), mk3(c), t, b1, b2)) t = FINF;
    const uint32_t orig = __float_as_uint(a.w);
    if (!(t > tmin)) return false;
    bool take = t < h.t;
    if (!take && t == h.t && h.pos >= 0) take = wins_tie(sc, (int)orig);
    if (!take) return false;
    h.t = t;
    h.prim = (int)orig;
    h.pos = cur;
    return ANY && any_hit;
  }

  template <class ST>
  PTD void begin(const DevScene& sc, v3 o_, v3 d_, float tmin_, float tmax, ST& st, uint32_t vseed_ = 0u,
                 float time_ = 0.f, bool any_hit_ = false) {
    h = HitOut{tmax, -1, -1};
    o = o_;
    d = d_;
    tmin = tmin_;
    time = time_;
    vseed = vseed_;
    any_hit = any_hit_;
    ro = o;
    rd = d;
    setup();
    moved = false;
    tr = TriRay{0, 0.f, 0.f, 0.f};
    cur = -1;
    base_sp = 0;
    enter_nodes(sc, sc.tlas_root);
    prim_base = 0;
    kind = 0;
    st.sp = 0;
    ref = 0u;
    have = true;
  }

  // Constants of node_fast for the ray (ro, rd): the reciprocal of each
  // component, at most 2^100 in magnitude (a zero component gives no inf - inf
  // with the scene's planes), and the two offsets.  Where that bound cuts the
  // reciprocal the planes move out by another 2^80 (1e-6 of a length unit): a
  // ray that runs within a slab never leaves it, also in the plane of a face at
  // 0, where the plane's distance and its margin are both zero.  An infinite
  // component has distances 0, as in the exact test; a NaN one has NaN
  // distances, which the minima and maxima pass over: that axis then rejects
  // nothing.
  //
  // The bound holds for directions whose largest component lies between 2^-60
  // and 2^100, as the renderer's do: its rays start with the camera's and
  // instances' scales and are normalised or nearly so at each bounce.  QUERY
  // brings directions outside 2^-40 .. 2^40 there by a power of two and keeps
  // all node distances in that scale; a caller's shorter directions (below
  // 1e-30) would otherwise lose the ratios of their components.
  PTD static float bound_rcp(float x, float& room) {
    const float r = __builtin_amdgcn_rcpf(x);
    room = fabsf(r) > 0x1p100f ? 0x1p80f : 0.f;
    const float m = __builtin_amdgcn_fmed3f(r, -0x1p100f, 0x1p100f);
    return x != x ? x : m;
  }
  PTD void setup() {
    if (KEEP_INV) rinv = mk3(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
    if (FAST) fast_setup();
  }
  PTD void fast_setup() {
    v3 u = rd;
    if (QUERY) {
      scale = 1.f;
      const uint32_t m = __float_as_uint(fmaxf(fmaxf(fabsf(rd.x), fabsf(rd.y)), fabsf(rd.z)));
      constexpr uint32_t LO = (127u - 40u) << 23, HI = (127u + 40u) << 23;
      if (m - LO > HI - LO && m != 0u && m < 0x7F800000u) {
        // the power of two of m, 2^-126 .. 2^126, and its reciprocal
        const uint32_t e = min(max(m & 0x7F800000u, 0x00800000u), 0x7E800000u);
        const float s = __uint_as_float(0x7F000000u - e);
        scale = __uint_as_float(e);
        u = mk3(rd.x * s, rd.y * s, rd.z * s);
      }
    }
    v3 room;
    finv = mk3(bound_rcp(u.x, room.x), bound_rcp(u.y, room.y), bound_rcp(u.z, room.z));
    const v3 a = mk3(ro.x * finv.x, ro.y * finv.y, ro.z * finv.z);
    const v3 e = mk3(__builtin_fmaf(fabsf(a.x), 0x1p-21f, room.x), __builtin_fmaf(fabsf(a.y), 0x1p-21f, room.y),
                     __builtin_fmaf(fabsf(a.z), 0x1p-21f, room.z));
    nb = mk3(-a.x - e.x, -a.y - e.y, -a.z - e.z);
    fb = mk3(e.x - a.x, e.y - a.y, e.z - a.z);
    sx = finv.x < 0.f ? 16u : 0u;
    sy = finv.y < 0.f ? 48u : 32u;
    sz = finv.z < 0.f ? 80u : 64u;
  }
  // a distance along the ray as node_fast counts it
  PTD float node_dist(float t) const { return QUERY ? t * scale : t; }

  // One internal node: the children the ray may enter, the nearest taken
  // next and the others on the stack, second nearest on top.
  //
  // A plane's distance is one fused multiply-add, plane * inv + (-o * inv),
  // the planes a component meets first (near) and last (far) picked by their
  // address; the exact test (slab_test) subtracts, multiplies and sorts the
  // two distances.  Rounding: with u = 2^-24, the reciprocal is off by 2 u,
  // o * inv by u, the offset's sum and the fma by u each, so a distance is
  // off by less than 6 u (|o inv| + |plane inv - o inv|).  The offsets move
  // every plane outward by 8 u |o inv| and the entry distance shrinks by 32 u
  // of itself, which also covers the exact test's own rounding: the children
  // taken are those of the exact test, and now and then one more, which holds
  // a nearer hit only where a primitive's own distance is rounded further than
  // its box.  The shrunk entry distance goes on the stack, where it is compared
  // with the hit found meanwhile: without the margin (it stood on the exit
  // distance once) it may lie a few u above a primitive's in the same plane,
  // and equal hits were lost.  Empty slots (inf planes) always
  // fail, or, for a ray of NaNs, lead to a leaf of no primitives.
  //
  // Sorted by a network of five exchanges, reference and distance stored
  // together, a node takes about 180 instructions where the exact test with
  // its ranking by pairwise comparisons takes 450.  4 M random rays in the
  // mesh scene 1.18 -> 0.96 ms, one 1080p frame of it 4.57 -> 4.0 ms, its
  // camera-ray launch at 96 spp 16.7 -> 15.6 ms and the next bounce 13.3 ->
  // 11.5 ms; the Cornell box, whose rays meet 2.3 nodes, is unchanged.
  PTD void exchange(float& ta, uint32_t& ra, float& tb, uint32_t& rb) {
    const bool s = tb < ta;
    const float t0 = s ? tb : ta, t1 = s ? ta : tb;
    const uint32_t r0 = s ? rb : ra, r1 = s ? ra : rb;
    ta = t0; tb = t1; ra = r0; rb = r1;
  }
  template <class ST>
  PTD void node_fast(const DevScene& sc, ST& st) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    f4 nx, ny, nz, fx, fy, fz;
    u4 cr;
    if constexpr (WIDE) {
      const uint64_t p = node_ptr + ((uint64_t)ref << 7);
      auto ld = [&](uint32_t k) { return *(const __attribute__((address_space(1))) f4*)(p | k); };
      nx = ld(sx); fx = ld(sx ^ 16u);
      ny = ld(sy); fy = ld(sy ^ 16u);
      nz = ld(sz); fz = ld(sz ^ 16u);
      cr = *(const __attribute__((address_space(1))) u4*)(p + 96u);
    } else {
      const char* b = reinterpret_cast<const char*>(sc.nodes);
      const uint32_t p = (node_base + ref) << 7;
      auto ld = [&](uint32_t k) { return *reinterpret_cast<const f4*>(b + (p | k)); };
      nx = ld(sx); fx = ld(sx ^ 16u);
      ny = ld(sy); fy = ld(sy ^ 16u);
      nz = ld(sz); fz = ld(sz ^ 16u);
      cr = *reinterpret_cast<const u4*>(b + (p | 96u));
    }
    const float lo = node_dist(tmin), hi = node_dist(h.t);
    auto slab = [&](float ax, float bx, float ay, float by, float az, float bz) {
      float tn = fmaxf(fmaxf(fmaxf(__builtin_fmaf(ax, finv.x, nb.x), __builtin_fmaf(ay, finv.y, nb.y)),
                             __builtin_fmaf(az, finv.z, nb.z)), lo);
      const float tf = fminf(fminf(fminf(__builtin_fmaf(bx, finv.x, fb.x), __builtin_fmaf(by, finv.y, fb.y)),
                                   __builtin_fmaf(bz, finv.z, fb.z)), hi);
      tn = __builtin_fmaf(fabsf(tn), -0x1p-19f, tn);
      return tn <= tf ? tn : FINF;
    };
    float t0 = slab(nx.x, fx.x, ny.x, fy.x, nz.x, fz.x), t1 = slab(nx.y, fx.y, ny.y, fy.y, nz.y, fz.y);
    float t2 = slab(nx.z, fx.z, ny.z, fy.z, nz.z, fz.z), t3 = slab(nx.w, fx.w, ny.w, fy.w, nz.w, fz.w);
    uint32_t r0 = cr.x, r1 = cr.y, r2 = cr.z, r3 = cr.w;
    exchange(t0, r0, t1, r1);
    exchange(t2, r2, t3, r3);
    exchange(t0, r0, t2, r2);
    exchange(t1, r1, t3, r3);
    exchange(t1, r1, t2, r2);
    ref = r0;
    have = t0 < FINF;
    if (st.room()) {
      if (t3 < FINF) st.push_lds(r3, t3);
      if (t2 < FINF) st.push_lds(r2, t2);
      if (t1 < FINF) st.push_lds(r1, t1);
    } else {
      if (t3 < FINF) { st.put(st.sp, r3, t3); st.sp++; }
      if (t2 < FINF) { st.put(st.sp, r2, t2); st.sp++; }
      if (t1 < FINF) { st.put(st.sp, r1, t1); st.sp++; }
    }
  }

  PTD void enter_nodes(const DevScene& sc, uint32_t base) {
    if (WIDE && FAST)
      node_ptr = (uint64_t)(const __attribute__((address_space(1))) char*)(const char*)sc.nodes + ((uint64_t)base << 7);
    else
      node_base = base;
  }

  PTD bool at_node() const { return have && !(ref & LEAF_BIT); }

  // the entry in hand, from the stack when there is none; false: the ray is
  // done
  template <class ST>
  PTD bool next(const DevScene& sc, ST& st) {
    while (!have) {
      if (cur >= 0 && st.sp == base_sp) {
        cur = -1;
        enter_nodes(sc, sc.tlas_root);
        if (moved) {
          ro = o; rd = d;
          setup();
        }
      }
      if (st.sp == 0) return false;
      float etn;
      st.pop(ref, etn);
      have = !(etn > (FAST ? node_dist(h.t) : h.t));
    }
    return true;
  }

  // One trip of every lane in it: an internal node, in scenes with meshes
  // again while at least NODE_LANES lanes are at one, then a leaf or instance
  // entry of the lanes that hold one.  Returns false once the ray is done.
  //
  // A triangle leaf (two tests) takes twice a node's instructions and an
  // instance entry as many; entered at once, they ran for the few lanes that
  // were at one while the others waited (13 of 64 lanes busy per instruction
  // after the first bounce).  Nodes first, the leaves of several lanes meet:
  // mesh still at 96 spp 64.0 -> 59.7 ms with 8 lanes (59.2 with 16, 59.9
  // with 32), 16 scenes in a batch 61.0 -> 58.9 (59.5, 60.4) ms, next-week
  // scene 3.65 -> 3.57 (3.61, 3.70) ms.  Scenes without meshes, whose leaves
  // are cheap and nodes few, lose by the extra vote: Cornell box 10.07 ->
  // 10.22 ms, random spheres 1.66 -> 1.70 ms.
  static constexpr int NODE_LANES = 8;
  template <class ST>
  PTD bool step(const DevScene& sc, ST& st, TraceCounts& cnt) {
    bool run;
    do {
      if (at_node()) node(sc, st, cnt);
      run = next(sc, st);
    } while (MESH && __popcll(__ballot(run && at_node())) >= NODE_LANES);
    if (!run || at_node()) return run;
    return leaf(sc, st, cnt);
  }

  // the leaf or instance entry in hand; false when an any-hit query ends here
  template <class ST>
  PTD bool leaf(const DevScene& sc, ST& st, TraceCounts& cnt) {
    have = false;
    uint32_t first = ref & 0x0FFFFFFFu;
    uint32_t count = (ref >> 28) & 7u;
    if (cur < 0) {
      if (count == 0) return true;  // an empty slot (a ray of NaNs, a stack overflow)
      // enter the instance at top-level position `first`
      const uint4* ir = gp(sc.insts) + (size_t)first * 8;
      float4 w0 = as_f4(ir[0]);
      float4 w1 = as_f4(ir[1]);
      float4 w2 = as_f4(ir[2]);
      uint4 info = ir[3];
      if (COUNT) cnt.insts++;
      enter_nodes(sc, info.x);
      prim_base = info.y;
      kind = info.z & 0xFFu;
      // the object-space ray is formed for every instance and kept where
      // the instance has a transform: formed behind a branch on that flag,
      // the matrix would be loaded only after the flag arrives (a second
      // memory round trip per instance entry)
      // (component selects: a select of whole structs keeps this state
      // in scratch memory)
      const bool xf = (info.z >> 8) != 0;
      const v3 xo = xf_point(w0, w1, w2, o), xd = xf_vector(w0, w1, w2, d);
      ro = mk3(xf ? xo.x : o.x, xf ? xo.y : o.y, xf ? xo.z : o.z);
      rd = mk3(xf ? xd.x : d.x, xf ? xd.y : d.y, xf ? xd.z : d.z);
      moved = xf;
      if (xf) setup();
      if (MESH && kind == PT_GEOM_MESH) tr = tri_setup(rd);
      cur = (int)first;
      base_sp = st.sp;
      ref = 0u;  // the bottom-level root, next
      have = true;
      return true;
    }
    if (MESH && kind == PT_GEOM_MESH) {
      // triangles two at a time: both records are loaded before either
      // test, one memory round trip per pair (a leaf holds up to 4); the
      // candidates are still offered in leaf order
      for (uint32_t k = 0; k < count; k += 2) {
        const uint32_t p0 = prim_base + first + k;
        const bool two = k + 1 < count;
        const uint32_t p1 = two ? p0 + 1 : p0;
        const float4 a0 = gp(sc.tri)[3 * p0], b0 = gp(sc.tri)[3 * p0 + 1], c0 = gp(sc.tri)[3 * p0 + 2];
        const float4 a1 = gp(sc.tri)[3 * p1], b1 = gp(sc.tri)[3 * p1 + 1], c1 = gp(sc.tri)[3 * p1 + 2];
        if (offer_tri(sc, a0, b0, c0, cnt)) return false;
        if (two && offer_tri(sc, a1, b1, c1, cnt)) return false;
      }
      return true;
    }
    for (uint32_t k = 0; k < count; k++) {
      uint32_t p = prim_base + first + k;
      if (COUNT) cnt.prims++;
      float t = FINF;
      uint32_t orig = 0xFFFFFFFFu;
      if (SPH && kind == PT_GEOM_SPHERES) {
        t = isect_sphere(gp(sc.sph)[p], ro, rd, tmin);
      } else if (RECT && kind == PT_GEOM_RECTS) {
        float4 A = gp(sc.rect)[2 * p], B = gp(sc.rect)[2 * p + 1];
        const int axis = (int)__float_as_uint(B.y);
        if (KEEP_INV) {
          t = isect_rect(A, B.x, axis, ro, rd, axis == 0 ? rinv.x : (axis == 1 ? rinv.y : rinv.z));
        } else {
          t = isect_rect(A, B.x, axis, ro, rd, 1.0f / (axis == 0 ? rd.x : (axis == 1 ? rd.y : rd.z)));
        }
        orig = __float_as_uint(B.w);
      } else if (BOX && kind == PT_GEOM_BOXES) {
        float4 lo = gp(sc.box)[2 * p], hi = gp(sc.box)[2 * p + 1];
        t = isect_box(mk3(lo), mk3(hi), ro, exact_inv(), tmin);
        orig = __float_as_uint(lo.w);
      } else if (EXT && kind == PT_GEOM_VOLUMES) {
        float4 A = gp(sc.vol)[2 * p], B = gp(sc.vol)[2 * p + 1];
        orig = __float_as_uint(B.w) & 0x7FFFFFFFu;
        t = isect_volume(A, B, ro, rd, tmin, vol_xi(vseed, orig, (uint32_t)inst_at(sc, cur)));
      } else if (EXT && kind == PT_GEOM_CYLINDERS) {
        float4 A = gp(sc.cyl)[2 * p], B = gp(sc.cyl)[2 * p + 1];
        orig = __float_as_uint(B.w);
        t = isect_cylinder(A, B, ro, rd, tmin);
      } else if (EXT && kind == PT_GEOM_MOVING_SPHERES) {
        float4 A = gp(sc.mov)[3 * p], B = gp(sc.mov)[3 * p + 1], C = gp(sc.mov)[3 * p + 2];
        v3 c = moving_center(A, B, C, time);
        orig = __float_as_uint(B.w);
        t = isect_sphere(make_float4(c.x, c.y, c.z, A.w), ro, rd, tmin);
      } else if (MESH) {
        float4 a = gp(sc.tri)[3 * p], b = gp(sc.tri)[3 * p + 1], c = gp(sc.tri)[3 * p + 2];
        float b1, b2;
        if (!tri_test(tr, ro, mk3(a), mk3(b), mk3(c), t, b1, b2)) t = FINF;
        orig = __float_as_uint(a.w);
      }
      if (!(t > tmin)) continue;
      bool take = t < h.t;
      if (!take && t == h.t && h.pos >= 0) {
        if (SPH && kind == PT_GEOM_SPHERES) orig = gp(sc.sph_idx)[p];
        take = wins_tie(sc, (int)orig);
      }
      if (take) {
        if (SPH && kind == PT_GEOM_SPHERES && orig == 0xFFFFFFFFu) orig = gp(sc.sph_idx)[p];
        h.t = t;
        h.prim = (int)orig;
        h.pos = cur;
        if (ANY && any_hit) return false;
      }
    }
    return true;
  }

  template <class ST>
  PTD void node(const DevScene& sc, ST& st, TraceCounts& cnt) {
    if constexpr (FAST) {
      node_fast(sc, st);
      return;
    }
    have = false;
    if (COUNT) cnt.nodes++;
    const uint4* nd = sc.nodes + (size_t)(node_base + ref) * 8;
    uint4 q0 = nd[0], q1 = nd[1], q2 = nd[2], q3 = nd[3], q4 = nd[4], q5 = nd[5], q6 = nd[6];
    const uint32_t lox[4] = {q0.x, q0.y, q0.z, q0.w}, hix[4] = {q1.x, q1.y, q1.z, q1.w};
    const uint32_t loy[4] = {q2.x, q2.y, q2.z, q2.w}, hiy[4] = {q3.x, q3.y, q3.z, q3.w};
    const uint32_t loz[4] = {q4.x, q4.y, q4.z, q4.w}, hiz[4] = {q5.x, q5.y, q5.z, q5.w};
    const uint32_t cref[4] = {q6.x, q6.y, q6.z, q6.w};
    float tn[4];
    // every slot's test runs and empty slots are masked afterwards: a test
    // behind a branch on the slot lets the compiler load that slot's planes
    // only after the child words arrive, a second memory round trip per node
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const float ts = slab_test(__uint_as_float(lox[c]), __uint_as_float(hix[c]), __uint_as_float(loy[c]),
                                 __uint_as_float(hiy[c]), __uint_as_float(loz[c]), __uint_as_float(hiz[c]), ro, rinv,
                                 tmin, h.t);
      tn[c] = cref[c] != EMPTY_REF ? ts : FINF;
    }
    // rank by (tn, slot): the nearest is taken next, the others go on the
    // stack with the second nearest on top
    int nh = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) nh += (tn[c] != FINF);
#pragma unroll
    for (int c = 0; c < 4; c++) {
      if (tn[c] == FINF) continue;
      int rank = 0;
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (e != c && tn[e] != FINF && (tn[e] < tn[c] || (tn[e] == tn[c] && e < c))) rank++;
      if (rank == 0) {
        // the cull a pop would apply (the slab test's far bound is 2^-22 loose)
        if (!(tn[c] > h.t)) {
          ref = cref[c];
          have = true;
        }
      } else {
        st.put(st.sp + nh - 1 - rank, cref[c], tn[c]);
      }
    }
    if (nh > 0) st.sp += nh - 1;
  }
};

template <bool COUNT, bool EXT = false, int KINDS = KIND_ALL, bool ANY = false, bool WIDE = false, class ST>
PTD HitOut trace_closest(const DevScene& sc, v3 o, v3 d, float tmin, float tmax, ST& st, TraceCounts& cnt,
                         uint32_t vseed = 0u, float time = 0.f, bool any_hit = false) {
  Tracer<COUNT, EXT, KINDS, ANY, WIDE> t;
  t.begin(sc, o, d, tmin, tmax, st, vseed, time, any_hit);
  for (uint32_t trips = 0; trips < TRIPS_MAX && t.step(sc, st, cnt); trips++) {
  }
  return t.h;
}

}  // namespace pt
