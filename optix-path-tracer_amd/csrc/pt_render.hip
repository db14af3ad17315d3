// pt_render.hip -- gfx950 kernels of the per-sample render path: query
// kernels behind pt_trace_closest / pt_trace_occluded and the wavefront
// integrator that replaces the OptiX megakernel (programs/raygen.cu:148-168
// renderPixel and :66-123 color, closest-hit programs of
// programs/materials/*.cu, miss programs, shadow any-hit).
//
// Wavefront, one bounce at a time over SoA path state in HBM:
//   [extend (depth 0: path start + camera rays) -> (material sort)
//    -> shade + shadow ray + connect]* -> accumulate
// Path sets are split into wave segments (pt_layout.hpp): each wave reads
// its own segment and compacts its survivors into its own segment of the
// next set with a ballot, so the bounce loop takes no global atomic.  The
// counts live in device memory, so a whole batch is enqueued without host
// synchronisation.
#include "pt_wave.hpp"

namespace pt {

// ------------------------------------------------------- query kernels
// EXT: volumes draw their free flight from the ray's index
//
// A wave's rays lie 64 at a time, grid stride apart.  64 at a time in
// lock-step, or (REFILL, scenes with meshes) each lane one ray after another,
// idle lanes taking the wave's next ones together (see k_extend): rays
// between random points meet 4 nodes on average and up to 88, so lock-step
// waits.  4 M random rays in the mesh scene 965 -> 546 us with 16 idle lanes
// (1: 542, 32: 548); up to 131072 rays, one group per wave, are unchanged.
constexpr int QUERY_REFILL = 16;
template <bool EXT, bool REFILL, class TR, class DONE>
PTD void trace_queries(const DevScene& sc, const pt_ray* __restrict__ rays, uint64_t n, Stack& st, TR& tr,
                       TraceCounts& c, DONE done) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  const uint64_t base = (uint64_t)blockIdx.x * BLOCK + (threadIdx.x & ~63u);
  uint64_t i = base + __lane_id();
  bool busy = i < n;
  auto take = [&]() {
    const float4* r4 = reinterpret_cast<const float4*>(rays + i);
    const float4 a = r4[0], b = r4[1];
    c = TraceCounts{0, 0, 0};
    tr.begin(sc, mk3(a), mk3(b), a.w, b.w, st, EXT ? query_vseed(i) : 0u);
  };
  if (!REFILL) {
    for (; i < n; i += stride) {
      take();
      for (uint32_t trips = 0; trips < TRIPS_MAX && tr.step(sc, st, c); trips++) {
      }
      done(i);
    }
    return;
  }
  if (busy) take();
  uint64_t row = base + stride;  // wave-uniform: the 64 rays being handed out
  uint32_t given = 0;            // of them, handed out
  uint32_t trips = 0;
  while (true) {
    const bool over = ++trips > TRIPS_MAX;
    if (busy && (!tr.step(sc, st, c) || over)) {
      done(i);
      busy = false;
    }
    const uint64_t idle = __ballot(!busy);
    if (row >= n) {
      if (idle == ~0ull) break;
    } else if (__popcll(idle) >= QUERY_REFILL) {
      if (!busy) {
        const uint32_t k = given + lane_rank(idle);
        i = row + (k >> 6) * stride + (k & 63u);
        busy = i < n;
        if (busy) take();
      }
      given += (uint32_t)__popcll(idle);
      row += (given >> 6) * stride;
      given &= 63u;
      trips = 0;
    }
  }
}

template <bool COUNT, bool EXT, bool REFILL, bool WIDE>
__global__ __launch_bounds__(BLOCK) void k_trace_closest(DevScene sc, const pt_ray* __restrict__ rays, uint64_t n,
                                                         pt_hit* __restrict__ hits, uint32_t* __restrict__ counts,
                                                         uint2* spill, uint32_t* overflow) {
  __shared__ uint2 s_stk[STK_LDS * BLOCK];
  Stack st = make_stack(s_stk, spill, overflow);
  Tracer<COUNT, EXT, KIND_ALL, false, WIDE, true> tr;
  TraceCounts c;
  trace_queries<EXT, REFILL>(sc, rays, n, st, tr, c, [&](uint64_t i) {
    const HitOut& h = tr.h;
    pt_hit out;
    out.t = h.pos >= 0 ? h.t : FINF;
    out.inst = h.pos >= 0 ? inst_at(sc, h.pos) : -1;
    out.prim = h.prim;
    out.reserved = 0;
    hits[i] = out;
    if (COUNT) {
      counts[3 * i + 0] = c.nodes;
      counts[3 * i + 1] = c.prims;
      counts[3 * i + 2] = c.insts;
    }
  });
}

template <bool COUNT, bool EXT, bool REFILL, bool WIDE>
__global__ __launch_bounds__(BLOCK) void k_trace_occluded(DevScene sc, const pt_ray* __restrict__ rays, uint64_t n,
                                                          uint8_t* __restrict__ occ, uint2* spill,
                                                          uint32_t* overflow) {
  __shared__ uint2 s_stk[STK_LDS * BLOCK];
  Stack st = make_stack(s_stk, spill, overflow);
  Tracer<COUNT, EXT, KIND_ALL, false, WIDE, true> tr;
  TraceCounts c;
  trace_queries<EXT, REFILL>(sc, rays, n, st, tr, c, [&](uint64_t i) {
    const HitOut& h = tr.h;
    uint8_t o = 0;
    if (h.pos >= 0) o = sc.mats[hit_material(sc, h.pos, h.prim)].type == PT_MAT_DIFFUSE_LIGHT ? 0 : 1;
    occ[i] = o;
  });
}

// ------------------------------------------------------ wavefront kernels
// Slot index of position p in a batch of nslots.  Slots come in 64-slot chunks
// (an 8 x 8 tile of pixels, coherent camera rays); the chunk index
// goes through a keyed 4-round Feistel permutation, cycle-walked into the Q
// full chunks, so that the chunks a wave owns come from all over the
// batch's frames and every wave keeps about the image-average share of
// surviving paths (with slot = position a wave would keep the same 64
// pixels in every frame, and the waves on the light would idle).  A partial
// last chunk keeps its place.
PTD uint32_t slot_of(uint32_t p, uint32_t nslots) {
  const uint32_t Q = nslots >> 6, q = p >> 6;
  if (Q < 2 || q >= Q) return p;
  int bits = 32 - __clz(Q - 1);  // 2^bits >= Q, made even
  bits += bits & 1;
  const int half = bits >> 1;
  const uint32_t mask = (1u << half) - 1u;
  uint32_t x = q;
  do {  // a permutation of [0, 2^bits): the walk from q < Q returns below Q
    uint32_t L = x >> half, R = x & mask;
    for (uint32_t r = 1; r <= 4; r++) {
      const uint32_t t = L ^ (mix32(R ^ (0x9E3779B9u * r)) & mask);
      L = R;
      R = t;
    }
    x = (L << half) | R;
  } while (x >= Q);
  return (x << 6) | (p & 63u);
}

// Pixel r of a frame in tile order: whole 8 x 8 tiles row by row, 64 pixels
// each, then the columns right of them and the rows above.  A wave's 64 camera
// rays start close together in both directions and meet fewer different nodes,
// triangles and texels than along 64 pixels of one row: mesh still at 96 spp,
// camera-ray launch 15.6 -> 12.1 ms and its shading 16.8 -> 14.9 ms.
PTD void tile_pixel(uint32_t r, uint32_t W, uint32_t H, uint32_t& x, uint32_t& y) {
  const uint32_t tw = W >> 3, th = H >> 3, whole = tw * th * 64u;
  if (r < whole) {
    const uint32_t t = r >> 6, ty = t / tw;
    x = (t - ty * tw) * 8u + (r & 7u);
    y = ty * 8u + ((r >> 3) & 7u);
    return;
  }
  uint32_t q = r - whole;
  const uint32_t cw = W & 7u, right = cw * th * 8u;
  const bool in_right = q < right;
  if (!in_right) q -= right;
  const uint32_t w = in_right ? cw : W;
  y = q / w;
  x = q - y * w + (in_right ? tw * 8u : 0u);
  y += in_right ? 0u : th * 8u;
}

// raygen.cu:148-168 renderPixel up to the first rtTrace, raygen.cu:50-64
// generateRay, raygen.cu:66-74 color() set-up.
// One camera path: slot s0 + launch index of pixel r of frame `frame` of the
// scene, at position p of state set 0; in a batch of scenes the RNG state's top byte
// is replaced by the scene index.  Returns the stored ray and its time.
struct PathStart {
  float4 o, d;
  float tm;
};
PTD PathStart start_path(const DevPaths& P, const RenderConsts& rc, uint32_t p, uint32_t s0, uint32_t frame,
                         uint32_t r, bool batch, uint32_t sid) {
  const PathState S = P.st[0];
  uint32_t x, y;
  // (radiance-cache batches keep row order: the order of the paths is that
  // of the training records)
  if (rc.flags & PT_FLAG_RADIANCE_CACHE) {
    y = r / rc.W;
    x = r - y * rc.W;
  } else {
    tile_pixel(r, rc.W, rc.H, x, y);
  }
  const uint32_t pix = rc.W * y + x, s = s0 + pix;
  uint32_t seed = tea64(pix, frame);
  float u = ((float)x + rnd(seed)) / (float)rc.W;
  float v = ((float)y + rnd(seed)) / (float)rc.H;
  const DevCamera& c = rc.cam;
  v3 cu = mk3(c.u[0], c.u[1], c.u[2]), cv = mk3(c.v[0], c.v[1], c.v[2]);
  v3 rd = c.lens_radius * random_in_unit_disk(seed);
  v3 lens = cu * rd.x + cv * rd.y;
  v3 origin = mk3(c.org[0], c.org[1], c.org[2]) + lens;
  v3 dir = mk3(c.llc[0], c.llc[1], c.llc[2]) + u * mk3(c.hor[0], c.hor[1], c.hor[2]) +
           v * mk3(c.ver[0], c.ver[1], c.ver[2]) - origin;
  // prd.time (raygen.cu:69); kept per slot when the scene has moving spheres
  const float tm = c.time0 + rnd(seed) * (c.time1 - c.time0);
  if (rc.store_time) P.ptime[s] = tm;
  const float4 o4 =
      make_float4(origin.x, origin.y, origin.z, __uint_as_float(batch ? ((seed & 0xFFFFFFu) | (sid << 24)) : seed));
  uint32_t dw = s;
  if ((rc.flags & PT_FLAG_RADIANCE_CACHE) && train_hash(pix, frame) < rc.cache.train_threshold) dw |= TRAIN_BIT;
  const float4 d4 = make_float4(dir.x, dir.y, dir.z, __uint_as_float(dw));
  S.o[p] = o4;
  S.d[p] = d4;
  P.result[s] = make_float4(0.f, 0.f, 0.f, __uint_as_float(rc.max_depth));
  return PathStart{o4, d4, tm};
}
PTD void reset_segments(const DevPaths& P, uint32_t n, const Seg& g) {
  if (__lane_id() == 0) {
    P.seg[g.w] = n;
    P.tseg[g.w] = 0u;
    P.qseg[g.w] = 0u;
  }
}

// material bucket of a hit: 0 = miss, 1 + material type otherwise
PTD uint32_t material_key(const DevScene& sc, float4 h) {
  int pos = __float_as_int(h.y);
  // the isotropic medium and the normal shader share the last bucket
  return pos < 0 ? 0u : 1u + (uint32_t)min(sc.mats[hit_material(sc, pos, __float_as_int(h.z))].type, 6);
}

// Closest-hit query of every live path (raygen.cu:77).  With SORT the
// material bucket of each hit is recorded and counted per wave and bucket.
//
// START (depth 0, in == 0): the query starts the nstart camera paths
// itself (raygen.cu:148-168, 50-74): position i of the dense state set 0
// is slot slot_of(i, nstart), its ray is stored for the shading pass and
// traced at once.  A batch of scenes (MULTI) finds the slot's item
// (scene and frame) in the BatchStart tables.  The path start is VALU-bound (the 64
// round seed hash) and the traversal latency-bound, so one launch hides
// most of the former under the latter.  A separate instantiation: the
// path-start code costs the traversal of the other depths a few spills.
// Occupancy target (waves per SIMD) of a closest-hit instantiation: bounce
// rays of one scene fit 5 waves without spills; the camera-ray kernels and
// those of a batch of scenes do at 4.  Spilled registers pass through the
// data path that the nodes come by: the camera rays at 5 (19 spills) and the
// other kernels without meshes at 6 (12 spills) took the Cornell box 10.5
// instead of 10.2 ms and the mesh still 67.3 instead of 65.1 ms; a batch of
// 16 scenes took 66.6 ms with both and its bounce rays at 5, 65.4 ms with the
// latter alone, 63.6 ms with neither.
template <int KINDS, bool START, bool WIDE>
constexpr int extend_waves() { return START || WIDE ? 4 : PT_EXTEND_WAVES; }
template <int KINDS>
constexpr int extend_stk() { return (KINDS & 8) ? STK_LDS_EXTEND : 12; }
template <bool COUNT, bool SORT, bool MULTI, bool EXT, int KINDS = KIND_ALL, bool START = false, bool WIDE = MULTI>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(extend_waves<KINDS, START, WIDE>(), 8))) void k_extend(
    DevScene sc0, DevPaths P, int in, float tmin, uint2* spill, uint64_t* stats, const DevScene* __restrict__ scenes,
    RenderConsts rc, uint32_t nstart, BatchStart bs) {
  constexpr int NS = extend_stk<KINDS>();
  __shared__ uint2 s_stk[NS * BLOCK];
  StackT<NS> st = make_stack<NS>(s_stk, spill, P.counters + CTR_STACK_OVERFLOW);
  const Seg g = my_seg(P);
  constexpr bool starts = START;
  uint32_t n;
  if (starts) {
    if (!MULTI && rc.frame_dev) rc.frame0 = *rc.frame_dev;  // replayed graphs take the batch's frame from memory
    n = dense_count(nstart, g);
    reset_segments(P, n, g);
  } else {
    n = seg_count(P, in, g);
  }
  const PathState S = P.st[in];
  uint32_t bc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  TraceCounts c{0, 0, 0};
  constexpr bool REFILL = PT_EXTEND_REFILL > 0 && !START && (KINDS & 8) != 0;
  if (REFILL) {
    // Bounce rays in scenes with meshes differ widely in length (the sky
    // after one node, a mesh after dozens): each lane keeps tracing paths
    // of the wave's segment one after another, and the idle lanes take the
    // next paths together once PT_EXTEND_REFILL of them wait (few ray
    // set-ups per refill).  Every path is traced exactly as alone, so hits
    // and counts do not depend on which lane takes it.  (Scenes of a few
    // primitives, whose rays are all short, run faster in lock-step: the
    // lanes' steps stay alike.)  In a batch of scenes each lane keeps its
    // scene (16 scenes 59.1 -> 58.7 ms per pass, and 57.8 ms with the node
    // array's address kept per ray and the table's pointers known as global).
    Tracer<COUNT, EXT, KINDS, false, WIDE> tr;
    uint32_t j = __lane_id(), sid = 0;
    auto scene = [&]() -> const DevScene& { return MULTI ? scenes[sid] : sc0; };
    bool busy = j < n;
    uint32_t next = 64;  // wave-uniform: the next position to hand out
    auto take = [&](uint32_t jj) {
      const uint32_t i = g.pos(jj);
      const float4 o = S.o[i], d = S.d[i];
      sid = __float_as_uint(o.w) >> 24;
      const float tm = (EXT && scene().mov_instances) ? P.ptime[__float_as_uint(d.w) & SLOT_MASK] : 0.f;
      tr.begin(scene(), mk3(o), mk3(d), tmin, FINF, st, __float_as_uint(o.w), tm);
    };
    if (busy) take(j);
    uint32_t trips = 0;
    while (true) {
      const bool over = ++trips > TRIPS_MAX;
      if (busy && (!tr.step(scene(), st, c) || over)) {
        P.hit[g.pos(j)] = make_float4(tr.h.t, __int_as_float(tr.h.pos), __int_as_float(tr.h.prim), 0.f);
        busy = false;
      }
      const uint64_t idle = __ballot(!busy);
      if (next >= n) {
        if (idle == ~0ull) break;
      } else if (__popcll(idle) >= (uint32_t)PT_EXTEND_REFILL) {
        if (!busy) {
          const uint32_t jn = next + lane_rank(idle);
          if (jn < n) {
            j = jn;
            take(j);
            busy = true;
          }
        }
        next += (uint32_t)__popcll(idle);
        trips = 0;
      }
    }
    if (SORT) {
      // material keys and bucket counts of the wave's hits, 64 at a time
      // (the material look-ups' latency paid once per 64 paths); the
      // fence makes the hits other lanes stored visible to these loads
      __threadfence_block();
      for (uint32_t j0 = 0; j0 < n; j0 += 64) {
        const uint32_t jj = j0 + __lane_id();
        uint32_t key = 0xFFu;
        if (jj < n) {
          const uint32_t i = g.pos(jj);
          key = material_key(MULTI ? scenes[__float_as_uint(S.o[i].w) >> 24] : sc0, P.hit[i]);
          P.keys[i] = key;
        }
#pragma unroll
        for (uint32_t b = 0; b < 8; b++) bc[b] += (uint32_t)__popcll(__ballot(key == b));
      }
    }
  }
  for (uint32_t j0 = 0; j0 < (REFILL ? 0u : n); j0 += 64) {
    const uint32_t j = j0 + __lane_id(), i = g.pos(j);
    uint32_t key = 0xFFu;
    if (j < n) {
      float4 o, d;
      float tm = 0.f;
      if (starts) {
        const uint32_t s = slot_of(i, nstart);
        PathStart ps;
        if (MULTI) {
          uint32_t lo = 0, hi = bs.nitems - 1;  // last item starting at or before s
          while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) >> 1;
            if (bs.off[mid] <= s) lo = mid;
            else hi = mid - 1;
          }
          const uint32_t sid = bs.scene[lo];
          ps = start_path(P, bs.rcs[sid], i, bs.off[lo], bs.frame[lo], s - bs.off[lo], true, sid);
        } else {
          const uint32_t f = s / rc.WH;
          ps = start_path(P, rc, i, f * rc.WH, rc.frame0 + f, s - f * rc.WH, false, 0u);
        }
        o = ps.o;
        d = ps.d;
        if (EXT && (MULTI || sc0.mov_instances)) tm = ps.tm;  // a batch's scenes differ: sc0 is the first one's
      } else {
        o = S.o[i];
        d = S.d[i];
      }
      const DevScene& sc = MULTI ? scenes[__float_as_uint(o.w) >> 24] : sc0;
      if (EXT && sc.mov_instances && !starts) tm = P.ptime[__float_as_uint(d.w) & SLOT_MASK];
      HitOut h = trace_closest<COUNT, EXT, KINDS, false, WIDE>(sc, mk3(o), mk3(d), tmin, FINF, st, c, __float_as_uint(o.w), tm);
      float4 hv = make_float4(h.t, __int_as_float(h.pos), __int_as_float(h.prim), 0.f);
      P.hit[i] = hv;
      if (SORT) {
        key = material_key(sc, hv);
        P.keys[i] = key;
      }
    }
    if (SORT) {
#pragma unroll
      for (uint32_t b = 0; b < 8; b++) bc[b] += (uint32_t)__popcll(__ballot(key == b));
    }
  }
  uint32_t a = c.nodes, b = c.prims, d = c.insts;
  if (COUNT) {
    for (int off = 32; off > 0; off >>= 1) {
      a += __shfl_down(a, off);
      b += __shfl_down(b, off);
      d += __shfl_down(d, off);
    }
  }
  if (__lane_id() == 0) {
    if (SORT) {
#pragma unroll
      for (int k = 0; k < 8; k++) P.bcount[(size_t)k * (gridDim.x * WAVES) + g.w] = bc[k];
    }
    stat_add(stats, g, STAT_EXT, n);
    if (COUNT) {
      stat_add(stats, g, STAT_NODES, a);
      stat_add(stats, g, STAT_PRIMS, b);
      stat_add(stats, g, STAT_INSTS, d);
    }
  }
}

// Exclusive scan of the (bucket, wave) counts in bucket-major order: the
// first sorted position of each wave's paths of each bucket, and the size
// of the sorted set.  The table holds 8 rows of `waves` entries (entry
// k * waves + w: bucket k of wave w, `waves` the launch grid's waves).
// Each of the block's 16 waves owns a contiguous chunk of whole 64-entry
// rows, read coalesced 16 loads at a time: a first pass sums the chunk,
// and after the chunk totals are exchanged a second pass (re-reading from
// L2) scans 64 entries at a time across the wave's lanes and writes the
// positions.
constexpr int SCAN_THREADS = 1024;
constexpr int SCAN_BATCH = 16;
__global__ __launch_bounds__(SCAN_THREADS) void k_sort_scan(DevPaths P, uint32_t waves) {
  constexpr int NW = SCAN_THREADS / 64;
  __shared__ uint32_t wsum[NW];
  const uint32_t lane = __lane_id(), wv = threadIdx.x >> 6;
  const uint32_t total = 8u * waves, rows = (total + 63u) / 64u;
  const uint32_t per = ((rows + NW - 1) / NW + SCAN_BATCH - 1) / SCAN_BATCH * SCAN_BATCH;  // rows per wave
  const uint32_t e0 = wv * per * 64u + lane;
  auto count = [&](uint32_t e) -> uint32_t { return e < total ? P.bcount[e] : 0u; };
  uint32_t sum = 0;
#pragma unroll 1
  for (uint32_t b0 = 0; b0 < per; b0 += SCAN_BATCH) {
    uint32_t v[SCAN_BATCH];
#pragma unroll
    for (int i = 0; i < SCAN_BATCH; i++) v[i] = count(e0 + 64u * (b0 + i));
#pragma unroll
    for (int i = 0; i < SCAN_BATCH; i++) sum += v[i];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if (lane == 0) wsum[wv] = sum;
  __syncthreads();
  uint32_t run = 0, all = 0;
#pragma unroll
  for (int k = 0; k < NW; k++) {
    const uint32_t t = wsum[k];
    run += (uint32_t)k < wv ? t : 0u;
    all += t;
  }
#pragma unroll 1
  for (uint32_t b0 = 0; b0 < per; b0 += SCAN_BATCH) {
    uint32_t v[SCAN_BATCH];
#pragma unroll
    for (int i = 0; i < SCAN_BATCH; i++) v[i] = count(e0 + 64u * (b0 + i));
#pragma unroll
    for (int i = 0; i < SCAN_BATCH; i++) {
      uint32_t s = v[i];
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(s, off);
        if (lane >= (uint32_t)off) s += t;
      }
      const uint32_t e = e0 + 64u * (b0 + i);
      if (e < total) P.bbase[e] = run + s - v[i];
      run += __shfl(s, 63);
    }
  }
  if (threadIdx.x == 0) P.counters[CTR_SORTED] = all;
}
// Move path state and hit into material-bucket order (state set 2, a dense
// set): each wave writes its bucket-b paths from its scanned base on.
__global__ __launch_bounds__(BLOCK) void k_sort_scatter(DevPaths P, int in) {
  const Seg g = my_seg(P);
  const uint32_t n = seg_count(P, in, g);
  const PathState S = P.st[in], D = P.st[2];
  uint32_t cur[8];
#pragma unroll
  for (int k = 0; k < 8; k++) cur[k] = uniform(P.bbase[(size_t)k * (gridDim.x * WAVES) + g.w]);
  for (uint32_t j0 = 0; j0 < n; j0 += 64) {
    const uint32_t j = j0 + __lane_id(), i = g.pos(j);
    const uint32_t key = j < n ? P.keys[i] : 0xFFu;
    uint32_t dst = 0;
#pragma unroll
    for (uint32_t b = 0; b < 8; b++) {
      const uint64_t m = __ballot(key == b);
      if (key == b) dst = cur[b] + lane_rank(m);
      cur[b] += (uint32_t)__popcll(m);
    }
    if (key < 8) {
      D.o[dst] = S.o[i];
      D.d[dst] = S.d[i];
      D.T[dst] = S.T[i];
      D.L[dst] = S.L[i];
      P.hit_sorted[dst] = P.hit[i];
    }
  }
  if (__lane_id() == 0) P.seg[2 * MAX_WAVES + g.w] = dense_count(P.counters[CTR_SORTED], g);
}

// Paths alive after the last bounce end with color() = 0 (raygen.cu:121-122);
// only their signature is recorded.
__global__ __launch_bounds__(BLOCK) void k_exhausted(DevPaths P, int in, uint64_t* stats) {
  const Seg g = my_seg(P);
  const uint32_t n = seg_count(P, in, g);
  const PathState S = P.st[in];
  if (__lane_id() == 0) stat_add(stats, g, STAT_EXHAUSTED, n);
  for (uint32_t j = __lane_id(); j < n; j += 64) {
    const uint32_t i = g.pos(j);
    P.sig_final[__float_as_uint(S.d[i].w) & SLOT_MASK] = __float_as_uint(S.L[i].w);
  }
}

// Sum of the per-wave statistics rows of a render (one block per word).
__global__ __launch_bounds__(BLOCK) void k_stats_reduce(const uint64_t* __restrict__ part, uint64_t* __restrict__ total) {
  __shared__ unsigned long long red[BLOCK];
  unsigned long long v = 0;
  for (uint32_t w = threadIdx.x; w < (uint32_t)MAX_WAVES; w += BLOCK) v += part[(size_t)w * STAT_WORDS + blockIdx.x];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int off = BLOCK / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) total[blockIdx.x] = red[0];
}

// Radiance-cache records after a batch: exclusive prefix sums of the
// per-wave training and query counts (waves of the batch's grid) and their
// totals.  One block of SCAN_THREADS threads.
__global__ __launch_bounds__(SCAN_THREADS) void k_cache_scan(DevPaths P, uint32_t waves) {
  __shared__ uint32_t part[SCAN_THREADS];
  const uint32_t per = (waves + SCAN_THREADS - 1) / SCAN_THREADS;
  const uint32_t e0 = min(threadIdx.x * per, waves), e1 = min(e0 + per, waves);
  for (int which = 0; which < 2; which++) {
    const uint32_t* cnt = which == 0 ? P.tseg : P.qseg;
    uint32_t* pre = which == 0 ? P.tpre : P.qpre;
    uint32_t sum = 0;
    for (uint32_t e = e0; e < e1; e++) sum += cnt[e];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < SCAN_THREADS; off <<= 1) {
      uint32_t v = threadIdx.x >= (uint32_t)off ? part[threadIdx.x - off] : 0u;
      __syncthreads();
      part[threadIdx.x] += v;
      __syncthreads();
    }
    uint32_t run = threadIdx.x ? part[threadIdx.x - 1] : 0u;
    for (uint32_t e = e0; e < e1; e++) {
      pre[e] = run;
      run += cnt[e];
    }
    if (threadIdx.x == SCAN_THREADS - 1) P.counters[which == 0 ? CTR_TRAIN : CTR_QUERY] = part[SCAN_THREADS - 1];
    __syncthreads();
  }
}

// Dense copies of `rows` records (which 0: training vertices, 1: queries)
// spread evenly over the batch's `total` records (all of them when rows ==
// total), row r taking the record of rank (r * mul) mod rows (mul coprime to
// rows: with mul ~ 0.618 rows every run of rows, such as one Adam batch,
// samples the whole image instead of a few waves' pixels): features, and
// for training vertices the target
//   radiance leaving the vertex toward the camera side
//     = (L_final - L_before) / T
// per channel, zero where T is zero or the value is not finite.  vals (9
// per row: L, T, target for training vertices; T, 0, network output for
// queries) and slots are optional.
__global__ __launch_bounds__(BLOCK) void k_cache_gather(DevPaths P, int which, uint32_t rows, uint32_t mul,
                                                        uint32_t half_step, uint32_t waves, uint32_t stride,
                                                        uint4* __restrict__ feat, float* __restrict__ tgt,
                                                        float* __restrict__ vals, uint32_t* __restrict__ slots) {
  const uint32_t total = P.counters[which == 0 ? CTR_TRAIN : CTR_QUERY];
  const uint32_t* pre = which == 0 ? P.tpre : P.qpre;
  // half_step = k: ranks move by total / (2 k) (records between those a
  // gather of k rows takes; the same ones when total < 2 k)
  const uint32_t shift = half_step ? total / (2u * half_step) : 0u;
  for (uint32_t r = blockIdx.x * BLOCK + threadIdx.x; r < rows && r < total; r += gridDim.x * BLOCK) {
    const uint32_t rank = (uint32_t)((uint64_t)r * mul % rows);
    uint32_t idx = rows >= total ? rank : (uint32_t)((uint64_t)rank * total / rows);
    idx = (uint32_t)(((uint64_t)idx + shift) % total);
    uint32_t lo = 0, hi = waves - 1;  // last wave whose prefix is <= idx
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (pre[mid] <= idx) lo = mid;
      else hi = mid - 1;
    }
    const uint32_t j = idx - pre[lo];
    const size_t k = (size_t)(j >> 6) * stride + (size_t)lo * 64 + (j & 63u);
    const uint4* src = (which == 0 ? P.t_feat : P.q_feat) + k * 12;
    for (int q = 0; q < 12; q++) feat[(size_t)r * 12 + q] = src[q];
    float out[9];
    uint32_t slot;
    if (which == 0) {
      const float4 a = P.t_L[k], t = P.t_T[k];
      slot = __float_as_uint(a.w) & SLOT_MASK;
      const float4 fin = P.result[slot];
      const float L0[3] = {a.x, a.y, a.z}, T0[3] = {t.x, t.y, t.z}, Lf[3] = {fin.x, fin.y, fin.z};
      for (int c = 0; c < 3; c++) {
        float v = T0[c] > 0.f ? (Lf[c] - L0[c]) / T0[c] : 0.f;
        v = (v > 0.f && v < 3.0e38f) ? v : 0.f;
        out[c] = L0[c];
        out[3 + c] = T0[c];
        out[6 + c] = v;
      }
      if (tgt)
        for (int c = 0; c < 3; c++) tgt[(size_t)r * 3 + c] = out[6 + c];
    } else {
      const float4 m = P.q_meta[k];
      slot = __float_as_uint(m.w) & SLOT_MASK;
      out[0] = m.x;
      out[1] = m.y;
      out[2] = m.z;
      out[3] = out[4] = out[5] = 0.f;
      for (int c = 0; c < 3; c++) out[6 + c] = P.q_out[k * 3 + c];
    }
    if (vals)
      for (int c = 0; c < 9; c++) vals[(size_t)r * 9 + c] = out[c];
    if (slots) slots[r] = slot;
  }
}

// The queries' answers: result += T * cache_radiance(y) per channel, over
// each wave's query segment (same grid as the batch).
__global__ __launch_bounds__(BLOCK) void k_cache_apply(DevPaths P) {
  const Seg g = my_seg(P);
  const uint32_t n = uniform(P.qseg[g.w]);
  for (uint32_t j = __lane_id(); j < n; j += 64) {
    const uint32_t i = g.pos(j);
    float4 m = P.q_meta[i];
    const uint32_t slot = __float_as_uint(m.w) & SLOT_MASK;
    const float y0 = cache_radiance(P.q_out[3 * (size_t)i]), y1 = cache_radiance(P.q_out[3 * (size_t)i + 1]),
                y2 = cache_radiance(P.q_out[3 * (size_t)i + 2]);
    float4 r = P.result[slot];
    r.x += m.x * y0;
    r.y += m.y * y1;
    r.z += m.z * y2;
    P.result[slot] = r;
  }
}

// The cache's per-batch judge, on n training vertices the plain tracer
// finished (vals: 9 per row, T at 3..5 and the unbiased radiance sample t
// at 6..8) and the network's outputs y for them:
//   res[0] = sum T^2 (cache_radiance(y) - t)^2   squared error the answers
//                                                would add to the image
//   res[1] = sum T^2 t^2                          the same for answering 0
//                                                (ending the paths there)
//   res[2] = outputs that are not finite
// per channel, summed in FP64 in a fixed order (one block).
__global__ __launch_bounds__(BLOCK) void k_cache_judge(const float* __restrict__ vals, const float* __restrict__ y,
                                                       uint32_t n, double* __restrict__ res) {
  __shared__ double s_num[BLOCK], s_den[BLOCK], s_bad[BLOCK];
  double num = 0.0, den = 0.0, bad = 0.0;
  for (uint32_t r = threadIdx.x; r < n; r += BLOCK) {
    for (int c = 0; c < 3; c++) {
      const float yc = y[3 * (size_t)r + c];
      const double T = vals[9 * (size_t)r + 3 + c], t = vals[9 * (size_t)r + 6 + c];
      if (!(fabsf(yc) <= 3.0e38f)) bad += 1.0;
      const double e = (double)cache_radiance(yc) - t;
      num += T * T * e * e;
      den += T * T * t * t;
    }
  }
  s_num[threadIdx.x] = num;
  s_den[threadIdx.x] = den;
  s_bad[threadIdx.x] = bad;
  __syncthreads();
  for (int off = BLOCK / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) {
      s_num[threadIdx.x] += s_num[threadIdx.x + off];
      s_den[threadIdx.x] += s_den[threadIdx.x + off];
      s_bad[threadIdx.x] += s_bad[threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    res[0] = s_num[0];
    res[1] = s_den[0];
    res[2] = s_bad[0];
  }
}

// raygen.cu:126-134 de_nan and raygen.cu:166 acc_buffer += (rgb, 1), in FP64
// and frame order; accumulation row 0 is the top of the image (raygen.cu:153).
// Paths with a NaN channel are counted into the wave's statistics row.
__global__ __launch_bounds__(BLOCK) void k_accumulate(DevPaths P, RenderConsts rc, uint32_t nframes, double* accum,
                                                      uint64_t* stats) {
  uint32_t nans = 0;
  for (uint32_t pix = blockIdx.x * BLOCK + threadIdx.x; pix < rc.WH; pix += gridDim.x * BLOCK) {
    uint32_t x = pix % rc.W, y = pix / rc.W;
    size_t o = 3 * ((size_t)(rc.H - 1 - y) * rc.W + x);
    double a0 = accum[o], a1 = accum[o + 1], a2 = accum[o + 2];
    for (uint32_t f = 0; f < nframes; f++) {
      float4 r = P.result[(size_t)f * rc.WH + pix];
      const bool ok = (r.x == r.x) & (r.y == r.y) & (r.z == r.z);
      nans += ok ? 0u : 1u;
      float cx = (r.x == r.x) ? r.x : 0.f, cy = (r.y == r.y) ? r.y : 0.f, cz = (r.z == r.z) ? r.z : 0.f;
      a0 += (double)cx;
      a1 += (double)cy;
      a2 += (double)cz;
    }
    accum[o] = a0;
    accum[o + 1] = a1;
    accum[o + 2] = a2;
  }
  for (int d = 32; d >= 1; d >>= 1) nans += __shfl_xor(nans, d);
  if (__lane_id() == 0) stat_add(stats, my_seg(P), STAT_NAN, nans);
}

// raygen.cu:136-146 make_Color on the FP64 accumulation
__global__ __launch_bounds__(BLOCK) void k_display(const double* accum, uint32_t npix, uint32_t frames,
                                                   uchar4* rgba) {
  for (uint32_t i = blockIdx.x * BLOCK + threadIdx.x; i < npix; i += gridDim.x * BLOCK) {
    unsigned char c[3];
    for (int k = 0; k < 3; k++) {
      float avg = (float)(accum[3 * (size_t)i + k] / (double)frames);
      float s = clampf(sqrtf(avg), 0.f, 1.f);
      c[k] = (unsigned char)(int)(255.99 * (double)s);
    }
    rgba[i] = make_uchar4(c[0], c[1], c[2], 255);
  }
}

__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (uint64_t)gridDim.x * BLOCK) p[i] = v;
}
// Packed triples (vertices, normals, triangle indices as the caller holds
// them) to the 16-byte records the kernels read.  HBM-bound, 28 B per triple:
// the mesh scene's 2 M triples take under 20 us, where widening them on the
// host and copying 16 B each took 10 ms.
__global__ __launch_bounds__(BLOCK) void k_widen3(const uint32_t* __restrict__ src, uint64_t n, uint4* __restrict__ dst) {
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (uint64_t)gridDim.x * BLOCK)
    dst[i] = make_uint4(src[3 * i], src[3 * i + 1], src[3 * i + 2], 0u);
}
__global__ void k_fill_f64(double* p, uint64_t n, double v) {
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (uint64_t)gridDim.x * BLOCK) p[i] = v;
}

// --------------------------------------------------------- host launchers
void launch_trace_closest(const DevScene& sc, const pt_ray* rays, uint64_t n, pt_hit* hits, uint32_t* counts,
                          uint2* spill, uint32_t* overflow, int grid, hipStream_t st) {
#define PT_TRACE(C, V, R, W)                                                                                       \
  hipLaunchKernelGGL((k_trace_closest<C, V, R, W>), dim3(grid), dim3(BLOCK), 0, st, sc, rays, n, hits, counts, spill, \
                     overflow)
  const bool vol = sc.ext_instances != 0, refill = (sc.kinds & 8u) != 0;
  if (counts) {
    if (vol) PT_TRACE(true, true, false, false);
    else PT_TRACE(true, false, false, false);
  } else if (sc.wide) {
    if (vol) PT_TRACE(false, true, false, true);
    else PT_TRACE(false, false, true, true);
  } else if (vol) {
    PT_TRACE(false, true, false, false);
  } else if (refill) {
    PT_TRACE(false, false, true, false);
  } else {
    PT_TRACE(false, false, false, false);
  }
#undef PT_TRACE
}
void launch_trace_occluded(const DevScene& sc, const pt_ray* rays, uint64_t n, uint8_t* occ, uint2* spill,
                           uint32_t* overflow, int grid, hipStream_t st) {
#define PT_OCC(V, R, W) \
  hipLaunchKernelGGL((k_trace_occluded<false, V, R, W>), dim3(grid), dim3(BLOCK), 0, st, sc, rays, n, occ, spill, overflow)
  const bool vol = sc.ext_instances != 0, refill = (sc.kinds & 8u) != 0;
  if (sc.wide) {
    if (vol) PT_OCC(true, false, true);
    else PT_OCC(false, true, true);
  } else if (vol) {
    PT_OCC(true, false, false);
  } else if (refill) {
    PT_OCC(false, true, false);
  } else {
    PT_OCC(false, false, false);
  }
#undef PT_OCC
}
__global__ void k_set_frame(uint32_t* f, uint32_t v) { *f = v; }
__global__ void k_next_frames(uint32_t* f, uint32_t step) { *f += step; }
void launch_set_frame(uint32_t* frame_dev, uint32_t value, hipStream_t st) {
  hipLaunchKernelGGL(k_set_frame, dim3(1), dim3(1), 0, st, frame_dev, value);
}
void launch_next_frames(uint32_t* frame_dev, uint32_t step, hipStream_t st) {
  hipLaunchKernelGGL(k_next_frames, dim3(1), dim3(1), 0, st, frame_dev, step);
}
// instantiation for the scene's kinds: rects + boxes (the Cornell box),
// rects + meshes (meshes on a ground rect), spheres, analytic, all
static int extend_kinds(uint32_t k) {
  if (k == 6u || k == 10u || k == 1u) return (int)k;
  if ((k & 8u) == 0) return 7;
  return KIND_ALL;
}
void launch_extend(const DevScene& sc, const DevPaths& P, int in, float tmin, uint2* spill, uint64_t* stats,
                   bool count_traversal, bool sort, int grid, hipStream_t st, const DevScene* scenes,
                   const RenderConsts* start, uint32_t nstart, bool multi_ext, const BatchStart* bstart) {
  const RenderConsts rc = start ? *start : RenderConsts{};
  const bool starts = start != nullptr && scenes == nullptr && nstart != 0;
  const bool bstarts = bstart != nullptr && scenes != nullptr && nstart != 0 && bstart->nitems != 0;
  const BatchStart bs = bstarts ? *bstart : BatchStart{};
#define PT_EXTEND(C, S, M, E, K, ST)                                                                                \
  hipLaunchKernelGGL((k_extend<C, S, M, E, K, ST>), dim3(grid), dim3(BLOCK), 0, st, sc, P, in, tmin, spill, stats, \
                     scenes, rc, nstart, bs)
#define PT_EXTEND4(M, E, K, ST)                                          \
  do {                                                                   \
    if (count_traversal && sort) PT_EXTEND(true, true, M, E, K, ST);     \
    else if (count_traversal) PT_EXTEND(true, false, M, E, K, ST);       \
    else if (sort) PT_EXTEND(false, true, M, E, K, ST);                  \
    else PT_EXTEND(false, false, M, E, K, ST);                           \
  } while (0)
// the camera-ray pass never sorts (camera hits are shaded in pixel order)
#define PT_EXTEND2(M, E, K, ST)                                     \
  do {                                                              \
    if (count_traversal) PT_EXTEND(true, false, M, E, K, ST);       \
    else PT_EXTEND(false, false, M, E, K, ST);                      \
  } while (0)
#define PT_EXTEND_KINDS(ST, X)                                                                           \
  do {                                                                                                   \
    if (sc.ext_instances != 0) { /* volumes, cylinders, moving spheres */                              \
      X(false, true, KIND_ALL, ST);                                                                      \
    } else {                                                                                             \
      switch (extend_kinds(sc.kinds)) {                                                                  \
        case 6: X(false, false, 6, ST); break;                                                           \
        case 10: X(false, false, 10, ST); break;                                                         \
        case 1: X(false, false, 1, ST); break;                                                           \
        case 7: X(false, false, 7, ST); break;                                                           \
        default: X(false, false, KIND_ALL, ST);                                                          \
      }                                                                                                  \
    }                                                                                                    \
  } while (0)
  // One scene of 4 GB of nodes or more (it has meshes: nothing else comes
  // near).  218 M triangles, 1080p at 8 spp: 32.1 ms with the counting kernels,
  // 28.3 ms with these; 4 M rays 4.84 -> 4.45 ms.
#define PT_EXTEND_WIDE(S, ST)                                                                                       \
  do {                                                                                                              \
    if (sc.ext_instances != 0)                                                                                      \
      hipLaunchKernelGGL((k_extend<false, S, false, true, KIND_ALL, ST, true>), dim3(grid), dim3(BLOCK), 0, st, sc, \
                         P, in, tmin, spill, stats, scenes, rc, nstart, bs);                                        \
    else                                                                                                            \
      hipLaunchKernelGGL((k_extend<false, S, false, false, KIND_ALL, ST, true>), dim3(grid), dim3(BLOCK), 0, st,    \
                         sc, P, in, tmin, spill, stats, scenes, rc, nstart, bs);                                    \
  } while (0)
  if (!scenes && sc.wide && !count_traversal) {
    if (starts) PT_EXTEND_WIDE(false, true);
    else if (sort) PT_EXTEND_WIDE(true, false);
    else PT_EXTEND_WIDE(false, false);
  } else if (bstarts && multi_ext) {
    PT_EXTEND2(true, true, KIND_ALL, true);
  } else if (bstarts) {
    PT_EXTEND2(true, false, KIND_ALL, true);
  } else if (scenes && multi_ext) {  // a batch holding volumes, cylinders or moving spheres
    PT_EXTEND4(true, true, KIND_ALL, false);
  } else if (scenes) {
    PT_EXTEND4(true, false, KIND_ALL, false);
  } else if (starts) {
    PT_EXTEND_KINDS(true, PT_EXTEND2);
  } else {
    PT_EXTEND_KINDS(false, PT_EXTEND4);
  }
#undef PT_EXTEND_WIDE
#undef PT_EXTEND_KINDS
#undef PT_EXTEND2
#undef PT_EXTEND4
#undef PT_EXTEND
}
void launch_sort(const DevPaths& P, int in, int grid, hipStream_t st) {
  hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(SCAN_THREADS), 0, st, P, (uint32_t)(grid * WAVES));
  hipLaunchKernelGGL(k_sort_scatter, dim3(grid), dim3(BLOCK), 0, st, P, in);
}
int shade_material_set(uint32_t types_mask) {
  if ((types_mask & ~(uint32_t)MS_DIFFUSE) == 0) return MS_DIFFUSE;
  if ((types_mask & ~(uint32_t)MS_SPHERES) == 0) return MS_SPHERES;
  if ((types_mask & ~(uint32_t)MS_ALL) == 0) return MS_ALL;
  return MS_FULL;
}
void launch_cache_scan(const DevPaths& P, int grid, hipStream_t st) {
  hipLaunchKernelGGL(k_cache_scan, dim3(1), dim3(SCAN_THREADS), 0, st, P, (uint32_t)(grid * WAVES));
}
void launch_cache_gather(const DevPaths& P, int which, uint32_t rows, uint32_t mul, int grid, uint4* feat, float* tgt,
                         float* vals, uint32_t* slots, hipStream_t st, uint32_t half_step) {
  const int g = (int)std::max<uint32_t>(1, std::min<uint32_t>((rows + BLOCK - 1) / BLOCK, 2048));
  hipLaunchKernelGGL(k_cache_gather, dim3(g), dim3(BLOCK), 0, st, P, which, rows, mul, half_step,
                     (uint32_t)(grid * WAVES), (uint32_t)(grid * BLOCK), feat, tgt, vals, slots);
}
void launch_cache_judge(const float* vals, const float* y, uint32_t n, double* res, hipStream_t st) {
  hipLaunchKernelGGL(k_cache_judge, dim3(1), dim3(BLOCK), 0, st, vals, y, n, res);
}
void launch_cache_apply(const DevPaths& P, int grid, hipStream_t st) {
  hipLaunchKernelGGL(k_cache_apply, dim3(grid), dim3(BLOCK), 0, st, P);
}
void launch_exhausted(const DevPaths& P, int in, uint64_t* stats, int grid, hipStream_t st) {
  hipLaunchKernelGGL(k_exhausted, dim3(grid), dim3(BLOCK), 0, st, P, in, stats);
}
void launch_stats_reduce(const uint64_t* part, uint64_t* total, hipStream_t st) {
  hipLaunchKernelGGL(k_stats_reduce, dim3(STAT_WORDS), dim3(BLOCK), 0, st, part, total);
}
void launch_accumulate(const DevPaths& P, const RenderConsts& rc, uint32_t nframes, double* accum, uint64_t* stats,
                       int grid, hipStream_t st) {
  hipLaunchKernelGGL(k_accumulate, dim3(grid), dim3(BLOCK), 0, st, P, rc, nframes, accum, stats);
}
void launch_display(const double* accum, uint32_t npix, uint32_t frames, uchar4* rgba, int grid, hipStream_t st) {
  hipLaunchKernelGGL(k_display, dim3(grid), dim3(BLOCK), 0, st, accum, npix, frames, rgba);
}
void launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t st) {
  int grid = (int)std::min<uint64_t>((n + BLOCK - 1) / BLOCK + 1, 1024);
  hipLaunchKernelGGL(k_fill_u32, dim3(grid), dim3(BLOCK), 0, st, p, n, v);
}
void launch_widen3(const uint32_t* src, uint64_t n, uint4* dst, hipStream_t st) {
  if (n == 0) return;
  const int grid = (int)std::min<uint64_t>((n + BLOCK - 1) / BLOCK, 4096);
  hipLaunchKernelGGL(k_widen3, dim3(grid), dim3(BLOCK), 0, st, src, n, dst);
}
void launch_fill_f64(double* p, uint64_t n, double v, hipStream_t st) {
  int grid = (int)std::min<uint64_t>((n + BLOCK - 1) / BLOCK + 1, 1024);
  hipLaunchKernelGGL(k_fill_f64, dim3(grid), dim3(BLOCK), 0, st, p, n, v);
}

}  // namespace pt
