// Device side of the LBVH traversal: ray state, slab and triangle tests, and
// the persistent per-wave loop shared by the standalone query kernels
// (trace_kernels.hip) and the batch kernel (batch_kernels.hip).
//
// Replaces the per-ray recursion of boxIntersect (accelerators.h:668-690)
// and the candidate loop of castRay (main.cpp:343-358): instead of collecting
// every candidate and then testing them, one lane owns one ray and walks the
// tree with a stack, nearer child first, culling boxes against the best hit
// so far. The result is the (t, primitive id) lexicographic minimum, i.e. the
// NONE loop of main.cpp:373-387 (lowest index wins ties).
#pragma once
#include <type_traits>

#include "rq_internal.h"

namespace rq {

// The launch's ray count, slice sizes and segments: from the kernel arguments,
// or computed here from a count read from device memory
// (TraceArgs::nrays_dev).
struct Schedule {
  uint32_t n, chunk, small, big, segs;
};
template <class Args>
__device__ inline Schedule schedule_of(const Args* a, uint32_t waves, uint32_t grid) {
  if (!a->nrays_dev) return Schedule{a->nrays, a->chunk, a->chunk_small, a->big_slices, a->segs};
  const uint32_t n = min(a->nrays, __builtin_amdgcn_readfirstlane(*a->nrays_dev));
  const SliceSchedule q = slice_schedule(n, trace_chunk(n, waves, a->chunk));
  return Schedule{n, q.chunk, q.small, q.big, trace_segs(q.total, waves, grid)};
}
__device__ inline uint32_t slice_begin(const Schedule& a, uint64_t s) {
  return s <= a.big ? (uint32_t)min(s * a.chunk, (uint64_t)a.n)
                    : (uint32_t)min((uint64_t)a.big * a.chunk + (s - a.big) * a.small,
                                    (uint64_t)a.n);
}

// The lane's number, computed here and now (volatile: a value that the walk
// would hold in a register, or spill, across all of its loops).
__device__ inline int lane_now() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}
// This lane's rank among the lanes of a wave mask.
__device__ inline uint32_t rank_in(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Where a wave takes its slices of the ray stream from: Src::next(b, e)
// returns the wave's next slice [b, e) of the rays, or false when there is
// none left for it. It is called with every lane of the wave active and its
// result is wave-uniform.
//
// The standalone kernels number the slices (chunk rays each for the first
// big_slices, then chunk_small) and deal them to segments (seg_slice): the
// w-th wave of a segment starts on the segment's slice w (no atomic), and
// takes its slice waves + k from the k-th add to the segment's 64-bit counter
// that is never reset (k = counter add - TraceArgs::ctr_base). When the waves'
// first slices cover the segment no wave touches the counter; otherwise each
// wave makes exactly one failing add and every later slice is one add, so the
// launch moves the counter by exactly the segment's number of slices, which
// the host adds to the base of the slot's next launch.
template <class Cold, int WPB>
struct QuerySlices {
  Cold cold;
  Schedule sc;
  uint32_t seg, index, waves;  // the segment, this wave's index in it, its waves
  bool first = true;
  __device__ QuerySlices(const Cold& c, uint32_t wave_in_block)
      : cold(c), sc(schedule_of(c(), gridDim.x * WPB, gridDim.x)), seg(seg_of(blockIdx.x, sc.segs)),
        index(seg_index(blockIdx.x, sc.segs) * WPB + wave_in_block),
        waves(seg_blocks(seg, sc.segs, gridDim.x) * WPB) {}
  __device__ bool next(uint32_t& b, uint32_t& e) {
    uint64_t s = index;
    if (!first) {
      if (slice_begin(sc, seg_slice(seg, sc.segs, waves)) >= sc.n) return false;  // first slices cover all
      const auto* c = cold();
      uint64_t k = 0;
      if ((threadIdx.x & 63u) == 0u) k = atomicAdd(c->counter + seg * COUNTER_STRIDE, 1ull);
      k = (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(k >> 32)) << 32 |
          __builtin_amdgcn_readfirstlane((uint32_t)k);
      s = k - c->ctr_base[seg] + waves;
    }
    first = false;
    s = seg_slice(seg, sc.segs, s);
    b = slice_begin(sc, s), e = slice_begin(sc, s + 1);
    return b < sc.n;
  }
};
// One block's waves share the n rays of an item, 64 at a time from a counter
// in LDS (or one wave has an item and a counter of its own).
struct ItemRays {
  uint32_t* ctr;
  uint32_t n;
  __device__ bool next(uint32_t& b, uint32_t& e) {
    uint32_t k = 0;
    if ((threadIdx.x & 63u) == 0u) k = atomicAdd(ctr, 64u);
    b = __builtin_amdgcn_readfirstlane(k);
    e = min(b + 64u, n);
    return b < n;
  }
};

struct RayState {
  float ox, oy, oz, dx, dy, dz;
  float ix, iy, iz;  // 1/d
  bool sx, sy, sz;   // sign bit of 1/d: the near plane of that axis is hi
  float tmin;
};

// Relative slack on the far bound: a triangle's rounded Möller–Trumbore t can
// fall a few ulps outside the exact box of its vertices (hits on edges and
// vertices); culling only beyond far * (1 + 2^-15) keeps every box that holds
// the brute-force closest hit.
constexpr float SLAB_SLACK = 1.000030517578125f;
// Sphere scenes: the reference's sphere test computes d2 = l.l - tca^2, whose
// cancellation at a distance L moves a grazing hit's t by up to about
// L * 2^-11 (and can accept a ray just outside the box); culling at the best
// hit with a 2^-9 relative slack keeps every box whose sphere's computed t
// can still beat the best hit.
constexpr float SPHERE_SLACK = 1.001953125f;
constexpr float TRI_ERROR = 0x1p-19f;  // (tri_doubt)
// Wide walk: a record is loaded at a byte offset node * 64 held in 32 bits (a
// scalar base plus one vector offset) while the node count stays at or below
// this; larger trees take 64-bit addresses.
constexpr uint32_t WIDE_SMALL_MAX_NODES = 1u << 25;

// Slab test (same operations and order as the oracle): near/far planes by
// the sign of 1/d, t = (plane - o) * (1/d). A zero direction component gives
// +-inf, or NaN with the origin on the plane, which the NaN-ignoring max
// (near) / min (far) read as "inside". Hit when near <= far * SLAB_SLACK.
__device__ inline bool slab(const float4& lo, const float4& hi, const RayState& r, float thi,
                            float slack, float& tn) {
  const float nx = ((r.sx ? hi.x : lo.x) - r.ox) * r.ix, fx = ((r.sx ? lo.x : hi.x) - r.ox) * r.ix;
  const float ny = ((r.sy ? hi.y : lo.y) - r.oy) * r.iy, fy = ((r.sy ? lo.y : hi.y) - r.oy) * r.iy;
  const float nz = ((r.sz ? hi.z : lo.z) - r.oz) * r.iz, fz = ((r.sz ? lo.z : hi.z) - r.oz) * r.iz;
  tn = fmaxf(fmaxf(nx, ny), fmaxf(nz, r.tmin));
  const float tf = fminf(fminf(fx, fy), fminf(fz, thi));
  return tn <= tf * slack;
}

// Whether a ray is too steep for the wide walk's short form of a plane's distance,
// (1024 + q) * (step / d) + (base - o) / d: the two parts are some thousand times
// the distance, and must both be finite and normal for every step a grid can have
// (2^-60 to 2^92), which holds for 1/d within 2^-60 and 2^20. Steep rays (parallel
// to an axis, or nearly; 1/d infinite, 0 or NaN) take ((1024 + q) * step +
// (base - o)) / d instead: 24 more multiplications a visit, and the exact walk's
// own reading of an infinite 1/d (a plane on the origin gives NaN, "inside"). They
// have a copy of the loop: a branch inside the one loop holds both forms'
// registers (48 meshes 1940 us, 1820 with the copy, 1815 without either). Rays
// along an axis over 1.3 M triangles, 1 M of them: 164 us, the short form 163.
__device__ inline bool steep(const RayState& r) {
  const float x = fabsf(r.ix), y = fabsf(r.iy), z = fabsf(r.iz);
  return !(fmaxf(fmaxf(x, y), z) <= 0x1p20f && fminf(fminf(x, y), z) >= 0x1p-60f);
}
// Four planes of a wide node on one axis, a byte each in q: (1024 + q) * si + bi,
// the distances with si = step / d and bi = (base - o) / d; STEEP, with si = step
// and bi = base - o, times i = 1/d.
typedef _Float16 Half2 __attribute__((ext_vector_type(2)));
template <bool STEEP>
__device__ inline float4 wide_planes(uint32_t q, float si, float bi, float i) {
  // 0x6400 | q is the half-precision 1024 + q
  const Half2 a = __builtin_bit_cast(Half2, __builtin_amdgcn_perm(0x64646464u, q, 0x04010400u));
  const Half2 b = __builtin_bit_cast(Half2, __builtin_amdgcn_perm(0x64646464u, q, 0x04030402u));
  const float4 p =
      make_float4(__builtin_fmaf((float)a[0], si, bi), __builtin_fmaf((float)a[1], si, bi),
                  __builtin_fmaf((float)b[0], si, bi), __builtin_fmaf((float)b[1], si, bi));
  return STEEP ? make_float4(p.x * i, p.y * i, p.z * i, p.w * i) : p;
}
// Slot test of a wide node: the last axis joins the interval [tn, tf] of the
// others; eps is the relative slack on the far bound.
__device__ inline bool slot_hit(float n, float f, float eps, float& tn, float tf) {
  tn = fmaxf(tn, n), tf = fminf(tf, f);
  return tn <= __builtin_fmaf(fabsf(tf), eps, tf);
}

__device__ inline void cas_pair(uint32_t& ka, int32_t& ca, uint32_t& kb, int32_t& cb) {
  const bool sw = kb < ka;
  const uint32_t k0 = sw ? kb : ka, k1 = sw ? ka : kb;
  const int32_t c0 = sw ? cb : ca, c1 = sw ? ca : cb;
  ka = k0, kb = k1, ca = c0, cb = c1;
}
// The same exchange for hit / miss keys (any hit): a miss before a hit swaps.
// The flags stay lane masks, so only the two link selects are vector work.
__device__ inline void cas_hit(bool& ha, int32_t& ca, bool& hb, int32_t& cb) {
  const bool sw = !ha && hb;
  const int32_t c0 = sw ? cb : ca, c1 = sw ? ca : cb;
  const bool h0 = ha || hb, h1 = ha && hb;
  ha = h0, hb = h1, ca = c0, cb = c1;
}

// Möller–Trumbore, main.cpp:137-162 (v_0 read as v0), t restricted to
// (tmin, tmax], tmax the ray's or the best hit so far (the caller tells a tie
// from an end). Dot products (x*x' + y*y') + z*z', no contraction. inv is
// 1 / the determinant.
__device__ inline bool mt(const TriRec& T, const RayState& r, float tmax, float& t, float& u,
                          float& v, float& inv) {
  const float px = r.dy * T.e2.z - r.dz * T.e2.y;
  const float py = r.dz * T.e2.x - r.dx * T.e2.z;
  const float pz = r.dx * T.e2.y - r.dy * T.e2.x;
  const float det = (T.e1.x * px + T.e1.y * py) + T.e1.z * pz;
  if (fabsf(det) < 1e-6f) return false;
  inv = 1.0f / det;
  const float tx = r.ox - T.v0.x, ty = r.oy - T.v0.y, tz = r.oz - T.v0.z;
  const float uu = ((tx * px + ty * py) + tz * pz) * inv;
  if (uu < 0.0f || uu > 1.0f) return false;
  const float qx = ty * T.e1.z - tz * T.e1.y;
  const float qy = tz * T.e1.x - tx * T.e1.z;
  const float qz = tx * T.e1.y - ty * T.e1.x;
  const float vv = ((r.dx * qx + r.dy * qy) + r.dz * qz) * inv;
  if (vv < 0.0f || uu + vv > 1.0f) return false;
  const float tt = ((T.e2.x * qx + T.e2.y * qy) + T.e2.z * qz) * inv;
  if (!(tt > r.tmin && tt <= tmax)) return false;
  t = tt, u = uu, v = vv;
  return true;
}

// Geometric ray-sphere test of the reference (accelerators.h:79-92): a centre
// behind the origin (tca < 0) or a miss distance beyond the radius rejects;
// otherwise t0 = tca - thc, t1 = tca + thc, and castRay takes t1 when t0 < 0
// (main.cpp:349-353). The reference accepts that t whatever its value (it is
// >= 0 once tca >= 0); here it must lie in [tmin, tmax], as above.
__device__ inline bool sphere_hit(const TriRec& S, const RayState& r, float tmax, float& t) {
  const float lx = S.v0.x - r.ox, ly = S.v0.y - r.oy, lz = S.v0.z - r.oz;
  const float tca = (lx * r.dx + ly * r.dy) + lz * r.dz;
  if (tca < 0.0f) return false;
  const float d2 = ((lx * lx + ly * ly) + lz * lz) - tca * tca;
  const float r2 = S.e1.y;
  if (d2 > r2) return false;
  const float thc = sqrtf(r2 - d2);
  const float t0 = tca - thc, t1 = tca + thc;
  const float tt = t0 < 0.0f ? t1 : t0;
  if (!(tt >= r.tmin && tt <= tmax)) return false;
  t = tt;
  return true;
}

// The primitive tests accept some rays that miss the primitive's box: the
// sphere test by the cancellation above, the triangle test by its own rounding.
// The answers are those for the rays that hit the box; a wide node's box on the
// grid is larger than the exact one, so the wide walk tests the exact one where
// the primitive test leaves a doubt. (A tree of one primitive has no node, and so
// no box.)
__device__ inline bool leaf_box(const float lo[3], const float hi[3], const RayState& r,
                                float tmax, float slack) {
  const float o[3] = {r.ox, r.oy, r.oz}, i[3] = {r.ix, r.iy, r.iz};
  float tn = r.tmin, tf = tmax;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const bool s = signbit(i[k]);
    tn = fmaxf(((s ? hi[k] : lo[k]) - o[k]) * i[k], tn);
    tf = fminf(((s ? lo[k] : hi[k]) - o[k]) * i[k], tf);
  }
  return tn <= tf * slack;
}
// Whether a triangle hit's rounding may have made it. With m the largest
// component of the edges, D of the direction, and the distance from the origin to
// the first vertex at most t D + m, u, v and 1 - u - v are within
// K D m (t D + 2 m) / det of the exact ones, and t within that times m / D. Where
// they lie further inside, and t is known to 2^-16, the exact line passes through
// the triangle, and the slab test of its box accepts that (its slack is 2^-15).
// K = 2^-19: a search for the largest errors found 12 * 2^-24 for u and v, 17 for
// 1 - u - v and 26 for t. 2.1 M camera rays take 246 us without this and 251 with it.
__device__ inline bool tri_doubt(const TriRec& T, const RayState& r, float t, float u, float v,
                                 float inv) {
  const float m = fmaxf(fmaxf(fmaxf(fabsf(T.e1.x), fabsf(T.e1.y)), fmaxf(fabsf(T.e1.z), fabsf(T.e2.x))),
                        fmaxf(fabsf(T.e2.y), fabsf(T.e2.z)));
  const float d = fmaxf(fmaxf(fabsf(r.dx), fabsf(r.dy)), fabsf(r.dz));
  const float h = (m * TRI_ERROR) * (__builtin_fmaf(t, d, m + m) * fabsf(inv));
  return !(fminf(fminf(u, v), 1.0f - (u + v)) > h * d && t > (h * 0x1p16f) * m);
}
// Its box, from the record: each plane within 2^-23 of its vertices' coordinates of
// the build's. The rays that meet the box with its planes drawn in by more than that
// meet the build's too; the few others are tested on the box in the leaf's parent.
__device__ inline bool tri_box(const TriRec& T, const RayState& r, float tmax) {
  const float v[3] = {T.v0.x, T.v0.y, T.v0.z}, e[3] = {T.e1.x, T.e1.y, T.e1.z},
              f[3] = {T.e2.x, T.e2.y, T.e2.z};
  float lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    lo[k] = v[k] + fminf(fminf(e[k], f[k]), 0.0f);
    hi[k] = v[k] + fmaxf(fmaxf(e[k], f[k]), 0.0f);
    const float in = fmaxf(fabsf(lo[k]), fabsf(hi[k])) * 0x1p-21f;
    lo[k] += in, hi[k] -= in;
  }
  return leaf_box(lo, hi, r, tmax, SLAB_SLACK);
}
// The box of leaf k of n as the binary nodes hold it.
struct LeafBoxes {
  const int32_t* parent;  // BuildBuffers::parent
  const NodeRec* nodes;
};
__device__ inline bool stored_box(const LeafBoxes& b, uint32_t n, int32_t k, const RayState& r,
                                  float tmax, float slack) {
  const uint32_t p = (uint32_t)b.parent[n - 1u + (uint32_t)k];
  const float4* q = reinterpret_cast<const float4*>(b.nodes + (p >> 1)) + 2u * (p & 1u);
  const float4 l = q[0], h = q[1];
  const float lo[3] = {l.x, l.y, l.z}, hi[3] = {h.x, h.y, h.z};
  return leaf_box(lo, hi, r, tmax, slack);
}
// A sphere leaf's box, as the build gives it (leaf_record).
__device__ inline bool sphere_box(const TriRec& S, const RayState& r) {
  const float c[3] = {S.v0.x, S.v0.y, S.v0.z};
  float lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) lo[k] = (c[k] - S.e1.x) + 0.0f, hi[k] = (c[k] + S.e1.x) + 0.0f;
  return leaf_box(lo, hi, r, INFINITY, SPHERE_SLACK);
}

// The wide records as a raw buffer resource (scalar registers): loads at a
// 32-bit offset from it need no 64-bit address arithmetic. Dword 3 selects
// the 32-bit data format that gfx9 buffer instructions require.
__device__ inline __amdgpu_buffer_rsrc_t wide_rsrc(const TraceArgs& a) {
  const uint64_t bytes = (uint64_t)a.nprims * sizeof(WideNode);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<WideNode*>(a.wide), (short)0,
                                           (int)(uint32_t)min(bytes, (uint64_t)0xFFFFFFFFu),
                                           0x00020000);
}
typedef uint32_t Row __attribute__((ext_vector_type(4)));
template <int AT>
__device__ inline Row row_load(__amdgpu_buffer_rsrc_t r, uint32_t voff) {
  return __builtin_bit_cast(Row, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, AT, 0));
}

// ---- rays walked by several lanes ---------------------------------------------
// Once SPLIT_IDLE lanes of a wave are idle and cannot be refilled, they take
// entries off the stacks of the lanes still walking and walk those subtrees of
// the same rays. Such a split ray has a slot in the wave's LDS: the smallest
// (t, primitive) found by any of its lanes as one 64-bit word (the bits of t,
// ordered as unsigned, above the primitive), which the lanes also cull with,
// and t, u, v of that hit. A lane's part ends when its stack is empty; the
// results are written from the slots once the whole wave is idle. The minimum
// does not depend on who walks what, so answers are the same.
// A ray's walk is a chain of dependent fetches, and the longest of a wave's 64
// (or the only one, in a small launch) sets the wave's time: 2.1 M camera
// rays 0.31 -> 0.25 ms with their copies, 1 M uniform rays in a soup 0.48 ->
// 0.40 ms closest and 0.38 -> 0.31 ms any hit. Rays that are short throughout
// pay for the code's presence: 8.3 M frame rays 0.69 -> 0.71 ms. 48 idle
// lanes: from 40 on the helpers' work costs as much as it saves, at 56 the
// gain on camera rays is a third less; sharing only from the 4th, 7th or 10th
// such step on loses 1 to 10 % on every kind of ray.
constexpr uint32_t SPLIT_IDLE = 48;
// Visits that a launch's only ray makes by itself first: one that ends within
// them does not fetch the helpers' code (a call on a sphere of 80 k triangles
// 27.8 us at 0, 26.4 at 20 or 32; in a soup of 22 k, where helpers pay, 26 / 30 /
// 33, and 34 without them).
constexpr uint32_t SINGLE_ALONE = 20;
// Full waves (64 rays a slice) over fewer primitives than this walk without help: few
// of their rays are long enough to pay for the helpers' code (300 k camera rays with and
// without, any hit and closest, us: 80 triangles 23.2 / 21.2 and 22.7 / 22.7, 320 29.3 /
// 30.0 and 31.1 / 30.5, 1 M of them 50.3 / 49.1 and 51.9 / 51.8, soup of 300 16.1 / 15.7
// and 16.7 / 16.4; past it, soup of 4000 54.0 / 54.7, a sphere of 5120 61.6 / 65.9).
constexpr uint32_t SHARE_MIN_PRIMS = 512;
constexpr uint32_t SPLIT_SLOTS = 16;  // split rays of a wave at a time
struct SplitSlots {
  unsigned long long key[SPLIT_SLOTS];  // ~0: no hit; any hit: 0 once there is one
  float tuv[SPLIT_SLOTS][3];
  uint32_t ray[SPLIT_SLOTS];
};
// One wave's lanes read what others of its lanes wrote: LDS accesses of a wave
// complete in order, volatile keeps them in the code's order.
typedef volatile __attribute__((address_space(3))) SplitSlots* Slots;
__device__ inline uint32_t ord_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float ord_float(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}
// (+ 0: hits at -0 and at 0 tie)
__device__ inline uint32_t hit_ord(float t) { return ord_bits(t + 0.0f); }
__device__ inline unsigned long long hit_key(float t, int32_t prim) {
  return (unsigned long long)hit_ord(t) << 32 | (uint32_t)prim;
}

// Persistent traversal loop of one wave. BLOCK threads per block; DEPTH stack entries
// per lane in LDS ([depth][lane], conflict-free), deeper entries in the global
// overflow area ([depth][thread]); TSTACK: entries carry their entry distance
// and a closest-hit pop skips entries now beyond the best hit (the box test
// redone against the current best). Leaves reached from a node are tested in
// the same loop iteration; the order of node visits and triangle tests is the
// canonical one unless TSTACK skips an entry. Rays are taken a slice at a time
// from src; the loop returns when it has none left for the wave and its lanes
// are idle.
// SPHERES: the leaves may be spheres (a.sphere); false compiles triangles only.
// WIDE: walk the 4-wide nodes (a.wide) instead of the binary ones: the slots
// a ray's box test accepts are visited nearest first (closest hit; any hit in
// slot order), the others pushed farthest first. Their boxes contain the
// binary nodes' and are tested with the same slack, so culling is at least as
// conservative as the binary walk and the result (the lexicographic minimum)
// is the same; visit order differs.
// ROWS, how the wide walk addresses a record: a tree of more than
// WIDE_SMALL_MAX_NODES nodes in 64 bits (ROWS_BIG), smaller ones by 32-bit
// offsets from the array's base (ROWS_SMALL); ROWS_ANY decides per launch
// inside one code path.
// cold() points at the arguments a ray needs only when it starts or ends. The
// query kernels read them again from the kernel's argument memory each time:
// as hoisted scalars they crowded out the walk's own (33 of them spilled to
// vector lanes, which held two registers and cost reads in the loop).
// cold.leaf_boxes() hands out the leaves' exact boxes, for the few doubtful hits.
constexpr int ROWS_SMALL = 0, ROWS_BIG = 1, ROWS_ANY = 2;
template <bool ANY, bool COUNT, int BLOCK, int DEPTH, bool TSTACK, bool SPHERES, bool WIDE,
          int ROWS, bool SHARE, class Src, class Cold>
__device__ inline void trace_loop_impl(const TraceArgs& a, const Cold& cold, Src& src,
                                       int32_t* s_node, float* s_tn, SplitSlots* slots) {
  // (a tree past 32-bit offsets keeps the walk without it)
  constexpr bool SPLIT = WIDE && SHARE && ROWS != ROWS_BIG;
  static_assert(!(WIDE && COUNT), "counted traversal walks the binary nodes");
  const bool big = ROWS == ROWS_ANY ? a.nprims > WIDE_SMALL_MAX_NODES : ROWS == ROWS_BIG;
  const int tid = threadIdx.x;
  const float slack = (SPHERES && a.sphere) ? SPHERE_SLACK : SLAB_SLACK;
  const float eps = slack - 1.0f;

  RayState r{};  // lanes that never take a ray still read their (unused) octant
  bool active = false;
  uint32_t cnext = 0, cend = 0;  // what is left of the wave's slice
  bool wave_out = false;         // there are no more slices for this wave
  uint32_t ray = 0;
  int32_t node = 0, best = -1;
  int sp = 0;  // stack entries; PENDING: the lane's result is not written yet
  constexpr int PENDING = -1;
  float bt = 0.0f, bu = 0.0f, bv = 0.0f;
  uint32_t vis = 0, tst = 0;

  // the slot of a ray that several lanes walk (-1: this lane's alone; read only
  // where lanes share), slots used
  int own;
  uint32_t nslots = 0;
  // steps that the wave makes without help when it could have some
  uint32_t alone = 0u;
  if (SPLIT && a.nrays == 1u) alone = SINGLE_ALONE;
  if (SPLIT && a.nprims < SHARE_MIN_PRIMS && a.chunk >= 64u) alone = ~0u;
  const Slots ss = (Slots)slots;

  auto write_hit = [&](uint32_t of, bool hit, int32_t prim, float t, float u, float v) {
    const auto c = cold();
    const uint32_t oi = c->out_index ? c->out_index[of] : of;
    if (ANY) {
      c->occ[oi] = hit ? 1 : 0;
    } else {
      c->prim[oi] = hit ? prim : -1;
      if (c->t) c->t[oi] = hit ? t : INFINITY;
      if (c->u) c->u[oi] = u;
      if (c->v) c->v[oi] = v;
    }
    if (COUNT) {
      c->visits[oi] = vis;
      c->tests[oi] = tst;
    }
  };
  // The lane's ray, or its part of a split ray, is walked to the end. The result
  // stays in the lane until the lane is needed again: written where each ray ended, it
  // took a wave a read of the output pointers and stores of its own for each length of
  // ray (300 k camera rays over 80 triangles 24.1 -> 22.7 us closest and 24.5 -> 23.3 any
  // hit, 2.1 M over 1.3 M 252 -> 244, 16.8 M uniform ones over 5.2 M 1446 -> 1360). The
  // stack's height marks it: as a lane mask it made scalars spill, and all was lost.
  auto finish = [&](auto split) {
    if (!decltype(split)::value) {
      sp = PENDING;
    } else {
      sp = own < 0 ? PENDING : 0;
      own = -1;
    }
    active = false;
  };
  auto flush = [&] {
    if (sp == PENDING) {
      write_hit(ray, best >= 0, best, bt, bu, bv);
      sp = 0;
    }
  };
  // Entry `at` (DEPTH or deeper) of thread t's stack in the overflow area.
  auto spilled = [&](int at, int t) -> int32_t* {
    const auto c = cold();
    return c->gstack +
           c->gwords * ((size_t)(at - DEPTH) * (gridDim.x * BLOCK) + blockIdx.x * BLOCK + t);
  };
  auto push = [&](int32_t c, float tn) {
    if (sp < DEPTH) {
      s_node[sp * BLOCK + tid] = c;
      if (TSTACK) s_tn[sp * BLOCK + tid] = tn;
    } else if (sp < DEPTH + (int)cold()->gdepth) {
      int32_t* g = spilled(sp, tid);
      g[0] = c;
      if (TSTACK) g[1] = __float_as_int(tn);
    } else {
      atomicOr(cold()->err, 1u);  // deeper than any LBVH of 30-bit codes: reported
      return;
    }
    ++sp;
  };
  // Pops the next entry into `node`; false when the stack is empty. The LDS
  // entry is read unconditionally (at a clamped depth) and replaced by the
  // overflow entry only past the LDS depth: with one read per branch the
  // compiler merges them into a generic (flat) load, which takes the vector
  // memory path and waits on both counters for every pop.
  auto pop = [&]() -> bool {
    while (sp > 0) {
      --sp;
      const int ls = min(sp, DEPTH - 1);
      node = s_node[ls * BLOCK + tid];
      float tn = TSTACK ? s_tn[ls * BLOCK + tid] : 0.0f;
      if (sp >= DEPTH) {
        const int32_t* g = spilled(sp, tid);
        node = g[0];
        if (TSTACK) tn = __int_as_float(g[1]);
      }
      if (!TSTACK || ANY || tn <= bt * slack) return true;
    }
    return false;
  };

  // A doubtful hit on triangle T, the leaf `node`: whether the ray meets its box up
  // to the ray's own end.
  auto exact_hit = [&](const TriRec& T) -> bool {
    const float tmax = cold()->rays.tmax[ray];
    return tri_box(T, r, tmax) || stored_box(cold.leaf_boxes(), a.nprims, ~node, r, tmax, slack);
  };

  for (;;) {
    flush();
    if (SPLIT && nslots != 0u && __ballot(active) == 0ull) {
      const int lane = lane_now();
      if (lane < (int)nslots) {
        const unsigned long long key = ss->key[lane];
        write_hit(ss->ray[lane], key != ~0ull, (int32_t)(uint32_t)key, ss->tuv[lane][0],
                  ss->tuv[lane][1], ss->tuv[lane][2]);
      }
      nslots = 0;
    }
    // ---- refill idle lanes from the wave's slice of the ray stream -------
    uint64_t m = __ballot(!active);
#pragma unroll 1
    for (int round = 0; round < 2 && m && !wave_out; ++round) {
      if (cnext >= cend && !src.next(cnext, cend)) {
        wave_out = true;
        break;
      }
      const uint32_t take = min((uint32_t)__popcll(m), cend - cnext);
      const uint32_t rank = rank_in(m);
      if (!active && rank < take) {
        const uint32_t rr = cnext + rank;
        const auto c = cold();
        ray = rr;
        r.ox = c->rays.ox[rr], r.oy = c->rays.oy[rr], r.oz = c->rays.oz[rr];
        r.dx = c->rays.dx[rr], r.dy = c->rays.dy[rr], r.dz = c->rays.dz[rr];
        r.tmin = c->rays.tmin[rr], bt = c->rays.tmax[rr];
        r.ix = 1.0f / r.dx, r.iy = 1.0f / r.dy, r.iz = 1.0f / r.dz;
        r.sx = signbit(r.ix), r.sy = signbit(r.iy), r.sz = signbit(r.iz);
        best = -1, bu = 0.0f, bv = 0.0f, vis = 0, tst = 0, sp = 0;
        node = a.nprims == 1 ? ~0 : 0;
        active = r.tmin < bt && a.nprims != 0;
        if (!active) write_hit(rr, false, -1, 0.0f, 0.0f, 0.0f);
      }
      cnext += take;
      m = __ballot(!active);
    }
    if (__ballot(active) == 0ull && wave_out) break;

    const __amdgpu_buffer_rsrc_t wrs = wide_rsrc(a);

    // Idle lanes join the rays still walked: the k-th entry from the top of the
    // j-th lane's stack goes to the (k * lanes + j)-th idle lane. Lanes whose
    // rays are not split yet get a slot each while there are any.
    auto share = [&](uint64_t idle, uint32_t nidle) {
      const bool fresh = active && sp > 0 && own < 0;
      const uint64_t fm = __ballot(fresh);
      if (fresh) {
        const uint32_t k = nslots + rank_in(fm);
        if (k < SPLIT_SLOTS) {
          own = (int)k;
          ss->key[k] = best >= 0 ? hit_key(bt, best) : ~0ull;
          ss->tuv[k][0] = bt, ss->tuv[k][1] = bu, ss->tuv[k][2] = bv;
          ss->ray[k] = ray;
        }
      }
      nslots = min(SPLIT_SLOTS, nslots + (uint32_t)__popcll(fm));
      const bool giver = active && sp > 0 && own >= 0;
      const uint64_t gm = __ballot(giver);
      if (gm == 0ull) return;
      const uint32_t givers = (uint32_t)__popcll(gm);  // < 64: some lanes are idle
      const float inv = 1.0f / (float)givers;
      const int lane = lane_now();
      const uint32_t j = rank_in(gm), rank = rank_in(idle);
      // lane j of the table: the j-th giver (lane 63 takes the rest)
      const int table = __builtin_amdgcn_ds_permute((giver ? (int)j : 63) * 4, lane);
      const uint32_t k = (uint32_t)(((float)rank + 0.5f) * inv);
      const int from = __builtin_amdgcn_ds_bpermute((int)(rank - k * givers) * 4, table);
      const int gsp = __shfl(sp, from, 64);
      const bool help = !active && (int)k < gsp;
      flush();
      auto take = [&](auto& x) {
        const auto y = __shfl(x, from, 64);
        if (help) x = y;
      };
      take(ray), take(own), take(bt), take(r.tmin);
      take(r.ox), take(r.oy), take(r.oz), take(r.dx), take(r.dy), take(r.dz);
      take(r.ix), take(r.iy), take(r.iz);
      r.sx = signbit(r.ix), r.sy = signbit(r.iy), r.sz = signbit(r.iz);
      if (help) {
        const int at = gsp - 1 - (int)k;
        node = s_node[min(at, DEPTH - 1) * BLOCK + (tid - lane + from)];
        if (at >= DEPTH) node = spilled(at, tid - lane + from)[0];
        best = -1, sp = 0;
        active = true;
      } else if (giver && nidle > j) {
        const int given = (int)(((float)(nidle - 1u - j) + 0.5f) * inv) + 1;
        sp -= min(sp, given);
      }
    };
    // ---- traverse until enough lanes are idle to be worth a refill, or, HELP,
    // with the idle lanes' help until all are (its own copy of the loop: the
    // slots' reads stay out of the other one); a wave with a steep ray takes a
    // third copy ---------------------------------------------------------------
    auto walk = [&](auto split, auto any_steep) {
      constexpr bool HELP = decltype(split)::value, STEEP = decltype(any_steep)::value;
      for (;;) {
        if (HELP && active && own >= 0) {  // what the ray's other lanes found
          const uint32_t hi = (uint32_t)(ss->key[own] >> 32);
          if (!ANY)
            bt = fminf(bt, ord_float(hi));  // (a NaN while there is no hit)
          else if (hi == 0u)
            finish(split);
        }
        if (WIDE && active && node >= 0) {
          Row r0, r1, r2, r3;
          if (!big) {
            const uint32_t off = (uint32_t)node * (uint32_t)sizeof(WideNode);
            r0 = row_load<0>(wrs, off), r1 = row_load<16>(wrs, off);
            r2 = row_load<32>(wrs, off), r3 = row_load<48>(wrs, off);
          } else {
            const Row* w = reinterpret_cast<const Row*>(a.wide + node);
            r0 = w[0], r1 = w[1], r2 = w[2], r3 = w[3];
          }
          const int4 ln = make_int4((int)r3[0], (int)r3[1], (int)r3[2], (int)r3[3]);
          // near / far planes by the direction's sign (hi is near when 1/d < 0),
          // two axes and then the third: the planes of all three at once would
          // hold eight registers more
          float t0, t1, t2, t3, f0, f1, f2, f3;
          {
            float sx = __uint_as_float(r0[3]), bx = __uint_as_float(r0[0]) - r.ox;
            float sy = __uint_as_float(r1[0]), by = __uint_as_float(r0[1]) - r.oy;
            if (!STEEP) sx *= r.ix, bx *= r.ix, sy *= r.iy, by *= r.iy;
            const float4 nx = wide_planes<STEEP>(r.sx ? r1[3] : r1[2], sx, bx, r.ix),
                         fx = wide_planes<STEEP>(r.sx ? r1[2] : r1[3], sx, bx, r.ix),
                         ny = wide_planes<STEEP>(r.sy ? r2[1] : r2[0], sy, by, r.iy),
                         fy = wide_planes<STEEP>(r.sy ? r2[0] : r2[1], sy, by, r.iy);
            t0 = fmaxf(fmaxf(nx.x, ny.x), r.tmin), f0 = fminf(fminf(fx.x, fy.x), bt);
            t1 = fmaxf(fmaxf(nx.y, ny.y), r.tmin), f1 = fminf(fminf(fx.y, fy.y), bt);
            t2 = fmaxf(fmaxf(nx.z, ny.z), r.tmin), f2 = fminf(fminf(fx.z, fy.z), bt);
            t3 = fmaxf(fmaxf(nx.w, ny.w), r.tmin), f3 = fminf(fminf(fx.w, fy.w), bt);
          }
          __builtin_amdgcn_sched_barrier(0);
          float sz = __uint_as_float(r1[1]), bz = __uint_as_float(r0[2]) - r.oz;
          if (!STEEP) sz *= r.iz, bz *= r.iz;
          const float4 nz = wide_planes<STEEP>(r.sz ? r2[3] : r2[2], sz, bz, r.iz),
                       fz = wide_planes<STEEP>(r.sz ? r2[2] : r2[3], sz, bz, r.iz);
          const bool h0 = slot_hit(nz.x, fz.x, eps, t0, f0) & (ln.x != 0);
          const bool h1 = slot_hit(nz.y, fz.y, eps, t1, f1) & (ln.y != 0);
          const bool h2 = slot_hit(nz.z, fz.z, eps, t2, f2) & (ln.z != 0);
          const bool h3 = slot_hit(nz.w, fz.w, eps, t3, f3) & (ln.w != 0);
          const int k = (int)h0 + (int)h1 + (int)h2 + (int)h3;
          // sort the slots by entry distance, misses last: a hit's key is its
          // distance's bits (ordered for tn >= +0, i.e. tmin >= 0; otherwise
          // only the visit order suffers), a miss's 0xFFFFFFFF. Any hit: hits
          // first, distances unused.
          auto key = [](bool h, float t) -> uint32_t {
            return h ? (ANY ? 0u : __float_as_uint(t)) : 0xFFFFFFFFu;
          };
          uint32_t k0, k1, k2, k3;
          int32_t c0 = ln.x, c1 = ln.y, c2 = ln.z, c3 = ln.w;
          if (ANY) {
            // the same network on the hit flags (every pushed entry is a hit,
            // key 0)
            bool g0 = h0, g1 = h1, g2 = h2, g3 = h3;
            cas_hit(g0, c0, g1, c1), cas_hit(g2, c2, g3, c3);
            cas_hit(g0, c0, g2, c2), cas_hit(g1, c1, g3, c3);
            cas_hit(g1, c1, g2, c2);
            k0 = k1 = k2 = k3 = 0u;
          } else {
            k0 = key(h0, t0), k1 = key(h1, t1), k2 = key(h2, t2), k3 = key(h3, t3);
            cas_pair(k0, c0, k1, c1), cas_pair(k2, c2, k3, c3);
            cas_pair(k0, c0, k2, c2), cas_pair(k1, c1, k3, c3);
            cas_pair(k1, c1, k2, c2);
          }
          if (k == 0) {
            if (!pop()) finish(split);
          } else {
            // push the k-1 farther hits, farthest deepest: entry sp+j holds
            // sorted slot k-1-j; with three LDS entries free all three are
            // written (entries above the new top are dead)
            if (k > 1 && sp + 3 <= DEPTH) {
              const int32_t e0 = k == 4 ? c3 : (k == 3 ? c2 : c1), e1 = k == 4 ? c2 : c1;
              s_node[sp * BLOCK + tid] = e0;
              s_node[(sp + 1) * BLOCK + tid] = e1;
              s_node[(sp + 2) * BLOCK + tid] = c1;
              if (TSTACK) {
                const uint32_t d0 = k == 4 ? k3 : (k == 3 ? k2 : k1), d1 = k == 4 ? k2 : k1;
                s_tn[sp * BLOCK + tid] = __uint_as_float(d0);
                s_tn[(sp + 1) * BLOCK + tid] = __uint_as_float(d1);
                s_tn[(sp + 2) * BLOCK + tid] = __uint_as_float(k1);
              }
              sp += k - 1;
            } else {
              if (k > 3) push(c3, __uint_as_float(k3));
              if (k > 2) push(c2, __uint_as_float(k2));
              if (k > 1) push(c1, __uint_as_float(k1));
            }
            node = c0;
          }
        } else if (!WIDE && active && node >= 0) {
          const float4* q = reinterpret_cast<const float4*>(a.nodes + node);
          const float4 lo0 = q[0], hi0 = q[1], lo1 = q[2], hi1 = q[3];
          if (COUNT) vis += 2;
          float tn0, tn1;
          const bool h0 = slab(lo0, hi0, r, bt, slack, tn0);
          const bool h1 = slab(lo1, hi1, r, bt, slack, tn1);
          const int32_t c0 = __float_as_int(lo0.w), c1 = __float_as_int(hi0.w);
          if (h0 && h1) {
            const bool swap = tn1 < tn0;
            push(swap ? c0 : c1, swap ? tn0 : tn1);
            node = swap ? c1 : c0;
          } else if (h0) {
            node = c0;
          } else if (h1) {
            node = c1;
          } else if (!pop()) {
            finish(split);
          }
        }
        // leaves reached from here are tested before the next node fetch
        while (active && node < 0) {
          const TriRec T = a.tris[~node];
          if (COUNT) ++tst;
          float t, u = 0.0f, v = 0.0f;
          bool done = false, hit;
          if (SPHERES && a.sphere) {
            hit = sphere_hit(T, r, bt, t) && (!WIDE || a.nprims < 2u || sphere_box(T, r));
          } else {
            float inv;
            hit = mt(T, r, bt, t, u, v, inv);
            if (WIDE && hit && tri_doubt(T, r, t, u, v, inv) && a.nprims > 1u)
              hit = exact_hit(T);
          }
          if (hit) {
            const int32_t prim = __float_as_int(T.v0.w);
            // t <= bt, which is the ray's open end until there is a hit
            if (HELP && own >= 0) {
              if (ANY) {
                if (t < bt) ss->key[own] = 0ull, done = true;
              } else if (t < bt || (uint32_t)(ss->key[own] >> 32) == hit_ord(t)) {
                const unsigned long long key = hit_key(t, prim);
                __hip_atomic_fetch_min(&slots->key[own], key, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
                if (ss->key[own] == key)
                  ss->tuv[own][0] = t, ss->tuv[own][1] = u, ss->tuv[own][2] = v;
                bt = t;
              }
            } else if (ANY) {
              if (t < bt) best = prim, done = true;
            } else if (t < bt || (best >= 0 && prim < best)) {
              best = prim, bt = t, bu = u, bv = v;
            }
          }
          if (done || !pop()) finish(split);
        }
        const uint64_t idle = __ballot(!active);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (nidle == 64u) break;
        if (!HELP) {
          if (!wave_out && nidle >= a.refill_idle) break;
          if (SPLIT && nidle >= SPLIT_IDLE) {
            if (alone == 0u) break;
            --alone;
          }
        } else if (nidle >= SPLIT_IDLE) {
          share(idle, nidle);
        }
      }
    };
    // (a wave with few rays from the start walks the second copy only: a small
    // launch pays for the code it fetches)
    auto sharing = [&] {
      const uint32_t nidle = (uint32_t)__popcll(__ballot(!active));
      return nidle >= SPLIT_IDLE && nidle != 64u && (wave_out || nidle < a.refill_idle);
    };
    const bool any_steep = WIDE && __ballot(active && steep(r)) != 0ull;
    if constexpr (SPLIT) {
      if (any_steep) {
        own = -1;
        walk(std::true_type{}, std::true_type{});
      }
      if (alone != 0u || !sharing()) walk(std::false_type{}, std::false_type{});
    } else {
      // (which branch is expected places the loops: 48 meshes 1906 us without, 1820 with)
      if (__builtin_expect(any_steep, 0))
        walk(std::false_type{}, std::integral_constant<bool, WIDE>{});
      else
        walk(std::false_type{}, std::false_type{});
    }
    if (SPLIT) {
      if (sharing()) {
        own = -1;
        walk(std::true_type{}, std::false_type{});
      }
    }
  }
}

// One code path for trees of any size (the batch and serving kernels, whose
// launches walk many trees). SHARE, idle lanes share the last rays (slots): a
// serving step's items are 256 rays of a block that waits for its longest one
// (a burst of 16 requests 1515 -> 1380 us with its copies); a batch run's waves
// refill from item to item, and the code's presence costs them 3 %.
template <bool ANY, bool COUNT, int BLOCK, int DEPTH, bool TSTACK, bool SPHERES, bool WIDE,
          bool SHARE, class Src, class Cold>
__device__ inline void trace_loop(const TraceArgs& a, const Cold& cold, Src& src, int32_t* s_node,
                                  float* s_tn, SplitSlots* slots = nullptr) {
  trace_loop_impl<ANY, COUNT, BLOCK, DEPTH, TSTACK, SPHERES, WIDE, ROWS_ANY, SHARE>(
      a, cold, src, s_node, s_tn, slots);
}
// A path per record addressing, chosen once per launch (the query kernels:
// one tree).
template <bool ANY, bool COUNT, int BLOCK, int DEPTH, bool TSTACK, bool WIDE, class Src, class Cold>
__device__ inline void trace_loop_split(const TraceArgs& a, const Cold& cold, Src& src,
                                        int32_t* s_node, float* s_tn, SplitSlots* slots) {
  if (WIDE && a.nprims > WIDE_SMALL_MAX_NODES)
    trace_loop_impl<ANY, COUNT, BLOCK, DEPTH, TSTACK, true, WIDE, ROWS_BIG, false>(
        a, cold, src, s_node, s_tn, slots);
  else
    trace_loop_impl<ANY, COUNT, BLOCK, DEPTH, TSTACK, true, WIDE, ROWS_SMALL, true>(
        a, cold, src, s_node, s_tn, slots);
}

}  // namespace rq
