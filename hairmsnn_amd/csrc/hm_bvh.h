// Device-side BVH view and traversal (closest hit and any hit).
//
// Layout in HBM: the tree is built binary (64-byte nodes holding both
// children's boxes) and then collapsed into four-wide nodes (BvhNodeWide)
// that traversal reads; segments are 32-byte records in leaf order. A child index >= 0 is an inner node, < 0 codes a leaf: a run of
// consecutive positions of the segment array (leaf_code).
//
// Traversal is one ray per lane (wave64). The stack's lowest kStackLds entries
// live in LDS, one column per lane (conflict-free), deeper entries spill to a
// per-thread global area sized from the wide tree's depth at build time.
#pragma once

#include "hm_common.h"
#include "hm_curve.h"
#include "hm_geom.h"

namespace hm {

struct BvhNode {
  float4 a;  // child0 lo.xyz, child0 hi.x
  float4 b;  // child0 hi.yz,  child1 lo.xy
  float4 c;  // child1 lo.z,   child1 hi.xyz
  int4 d;    // child0, child1, unused, unused
};

// Four-wide node of 64 bytes: the children's boxes as 8-bit steps from the
// node's corner (plane = o + q * s per axis, child k in byte k of each word),
// rounded outward with a margin that covers the arithmetic of node_boxes
// (after the compressed wide nodes of Ylitie, Karras and Laine 2017, with
// FP32 steps instead of powers of two: the steps are as fine as 8 bits allow).
// child[k] >= 0 is an inner node, < 0 codes a leaf (leaf_code). An unused slot
// has an inverted box, which a ray practically never enters; its child code is
// leaf 0, so that a ray that does only tests a primitive that exists.
//
// Why 64 bytes: the vector memory path takes one 16-byte access of one lane
// per clock and CU when every lane reads a node of its own, whatever the
// occupancy. Chains of dependent node reads over 2^18 / 2^20 nodes measured
// 84 / 83 G nodes/s with 128-byte FP32 nodes (seven accesses) and 194 / 159
// with 64-byte ones (four).
constexpr int kBvhWidth = 4;
struct __attribute__((aligned(64))) BvhNodeWide {
  float ox, oy, oz, sx;
  float sy, sz;
  unsigned lox, hix, loy, hiy, loz, hiz;
  int child[kBvhWidth];
};
static_assert(sizeof(BvhNodeWide) == 64, "half a cache line per node");
constexpr int kEmptyChild = ~0;

struct BvhView {
  const BvhNodeWide* nodes;  // wide tree, root at 0
  const float4* segs;     // 2 float4 per segment: (p0, r), (p1, id bits)
  int num_segs;
};

struct SphereView {
  int enabled;
  float cx, cy, cz, r;
};

// OBJ head mesh: BVH over the triangles' boxes, vertices (3 float4 per
// triangle) for intersection, and per triangle 3 vertex normals + the diffuse
// colour (4 float4) for shading.
struct MeshView {
  BvhView bvh;
  const float4* tri;
  const float4* shade;
  int num;
};

// Stack entries per lane kept in LDS (4 bytes x 256 lanes each per block).
constexpr int kStackLds = 16;
constexpr int kTraceBlock = 256;
// Blocks per CU of a ray stream's grid. Each lane should get several rays, or
// a wave has nothing to refill from: a million rays over 8, 6, 4, 3 and 2
// blocks per CU measured 636, 659, 525, 535 and 679 us.
constexpr int kRayBlocksPerCu = 4;

// Launch bounds of the traversal kernels: 256 threads and a floor of waves per
// SIMD, which sets the register budget. Segments: 8 (the ray streams launch
// four waves per SIMD, so that two streams' launches run side by side); the
// round-curve iteration needs more registers.
#define HM_TRACE_BOUNDS_T(curves) __launch_bounds__(kTraceBlock, (curves) ? 4 : 8)

struct TraceCounters {
  uint32_t nodes;
  uint32_t segs;
  uint32_t rays;
};

#if defined(__HIPCC__)

struct RayInv {
  float ox, oy, oz, dx, dy, dz;
  float ix, iy, iz, oix, oiy, oiz;
};

HM_D float safe_inv(float d) {
  const float e = 1e-20f;
  return 1.f / (fabsf(d) > e ? d : copysignf(e, d));
}

HM_D RayInv make_ray(float ox, float oy, float oz, float dx, float dy, float dz) {
  RayInv r;
  r.ox = ox; r.oy = oy; r.oz = oz;
  r.dx = dx; r.dy = dy; r.dz = dz;
  r.ix = safe_inv(dx); r.iy = safe_inv(dy); r.iz = safe_inv(dz);
  r.oix = ox * r.ix; r.oiy = oy * r.iy; r.oiz = oz * r.iz;
  return r;
}

typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) int lds_int;

// Traversal stack of one lane: kStackLds entries in LDS, entry k of lane
// thread t of the block at byte 1024 k + 4 t (conflict-free), then
// spill_levels entries in memory. The LDS pointer keeps its address space,
// so the accesses are LDS instructions (through a generic pointer they were
// flat ones, which go through the vector memory path that the node loads
// need).
struct TraceStack {
  static constexpr int kLevel = kTraceBlock * (int)sizeof(int);
  lds_char* lds;     // the block's stacks
  int off;           // byte offset of the lane's next free entry
  int* spill;        // this thread's spill column
  int spill_stride;
  int spill_levels;
  HM_D void init(int* block_stacks, int* spill_column, int stride, int levels) {
    lds = (lds_char*)block_stacks;
    off = 4 * (int)threadIdx.x;
    spill = spill_column;
    spill_stride = stride;
    spill_levels = levels;
  }
  HM_D void clear() { off &= kLevel - 1; }
  HM_D bool empty() const { return off < kLevel; }
  HM_D lds_int* at(int o) const { return (lds_int*)(lds + o); }
  // Whether every active lane has room for three more entries in LDS (and
  // none in memory), decided for the whole wave.
  HM_D bool room3() const { return __ballot(off >= kLevel * (kStackLds - 2)) == 0; }
  // Writes v to the next entry and keeps it if `keep` (room3 holds).
  HM_D void put(int v, bool keep) {
    *at(off) = v;
    off += keep ? kLevel : 0;
  }
  HM_D void push(int v) {
    const int k = off / kLevel;
    if (k < kStackLds) *at(off) = v;
    else if (k - kStackLds < spill_levels) spill[(size_t)(k - kStackLds) * spill_stride] = v;
    else return;  // unreachable for a tree within the sized depth; drop rather than overrun
    off += kLevel;
  }
  HM_D int pop() {
    off -= kLevel;
    const int k = off / kLevel;
    return k < kStackLds ? *at(off) : spill[(size_t)(k - kStackLds) * spill_stride];
  }
  HM_D int pop_lds() {
    off -= kLevel;
    return *at(off);
  }
};

// Traversal: the current entry is an inner node (>= 0) or a leaf (~index <
// 0); a step either visits one wide node (nearest hit child next, the other
// hit children pushed far to near, leaves included) or tests one primitive.
constexpr int kNone = 0x7fffffff;

// One axis of a node against a ray (near and far planes picked by the sign of
// the direction, so no plane needs a min or max): the distances of the children's near and
// far planes are q * step + near / far. The corner's distance is widened by
// 2^-22 of itself on both sides, four times the rounding of its terms.
struct AxisSlabs {
  float step, near, far;
  unsigned qn, qf;  // near and far planes, one byte per child
  HM_D AxisSlabs(float o, float s, unsigned lo, unsigned hi, float inv, float oinv) {
    const float w = 2.384185791015625e-7f;
    step = s * inv;
    const float b = fmaf(o, inv, -oinv);
    near = fmaf(-fabsf(b), w, b);
    far = fmaf(fabsf(b), w, b);
    qn = inv < 0.f ? hi : lo;
    qf = inv < 0.f ? lo : hi;
  }
  HM_D float enter(int k) const { return fmaf((float)((qn >> (8 * k)) & 255u), step, near); }
  HM_D float leave(int k) const { return fmaf((float)((qf >> (8 * k)) & 255u), step, far); }
};

// A node's children and the entry distances of their boxes against
// [0, tmax]; t[k] is +inf where the ray misses child k.
HM_D void node_boxes(const BvhView& bvh, const RayInv& r, int node, float tmax, float t[4], int c[4]) {
  const int4* p = (const int4*)((const char*)bvh.nodes + (unsigned)node * (unsigned)sizeof(BvhNodeWide));
  const int4 a = p[0], b = p[1], d = p[2], ch = p[3];
  const AxisSlabs x(__int_as_float(a.x), __int_as_float(a.w), (unsigned)b.z, (unsigned)b.w, r.ix, r.oix);
  const AxisSlabs y(__int_as_float(a.y), __int_as_float(b.x), (unsigned)d.x, (unsigned)d.y, r.iy, r.oiy);
  const AxisSlabs z(__int_as_float(a.z), __int_as_float(b.y), (unsigned)d.z, (unsigned)d.w, r.iz, r.oiz);
  c[0] = ch.x; c[1] = ch.y; c[2] = ch.z; c[3] = ch.w;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float tn = fmaxf(fmaxf(x.enter(k), y.enter(k)), fmaxf(z.enter(k), 0.f));
    const float tf = fminf(fminf(x.leave(k), y.leave(k)), fminf(z.leave(k), tmax));
    t[k] = tn <= tf ? tn : __builtin_inff();
  }
}

// (entry distance, child) as one 64-bit value whose order as a double is
// the order of the distances: a non-negative float's bits in the high word
// make a non-negative finite double. One v_min_f64 / v_max_f64 (full rate on
// CDNA) then moves distance and child together; comparing and selecting the
// two words separately took five instructions per exchange instead of two.
HM_D double hit_key(float t, int c) { return __hiloint2double(__float_as_int(t), c); }
HM_D bool key_hit(double k) { return __int_as_float(__double2hiint(k)) < __builtin_inff(); }
HM_D int key_child(double k) { return __double2loint(k); }
HM_D void key_swap(double& a, double& b) {
  double lo, hi;
  asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
  asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
  a = lo;
  b = hi;
}

// Per-lane traversal state, advanced one step (one wide node or one
// primitive) at a time.
struct ClosestState {
  float best_t, best_u;
  int best_id;
  int cur;   // current entry: node (>= 0), ~leaf (< 0) or kNone when done
};

// Steps after which a query of a valid tree has certainly ended (each node and
// leaf is visited at most once); bounds the loops for a malformed tree.
HM_D int trace_cap(const BvhView& bvh) { return 2 * bvh.num_segs + 64; }

// Starts a closest-hit query with (best_t, best_id) preset by the caller
// (e.g. a hit on the head sphere).
HM_D void closest_begin(const BvhView& bvh, TraceStack& st, ClosestState& s) {
  st.clear();
  s.cur = bvh.num_segs > 0 ? 0 : kNone;
}

// Leaf tests: a leaf record is two float4s in Morton order whose second w
// holds the primitive id. Hair: the record is the segment itself. Triangle
// meshes: the record holds the triangle's box, the vertices are read by id.
//
// For the ray streams: a wave tests primitives when kPrims x (lanes waiting at
// a primitive) >= kNodes x (lanes waiting at a node), and takes its rays in
// chunks of kChunk. A segment test costs about a node step: a third of the
// lanes at segments is worth it (shares 1/2, 1/4 and 1/8 of the node lanes:
// 352, 357 and 375 us on a million mixed rays; 86.4, 88.8 and 93.7 ms on 16
// passes of the headline frame). A round curve's iteration costs an order of
// magnitude more, so two thirds of the lanes are waited for; and its rays
// differ so much that a wave's share is dealt out in small chunks.
struct SegLeaf {
  static constexpr int kPrims = 2, kNodes = 1, kChunk = 32;
  HM_D bool operator()(const BvhView& bvh, const RayInv& r, int leaf, float* t, float* u, int* id) const {
    const float4 s0 = bvh.segs[2 * leaf];
    const float4 s1 = bvh.segs[2 * leaf + 1];
    *id = __float_as_int(s1.w);
    return intersect_segment(r.ox, r.oy, r.oz, r.dx, r.dy, r.dz, s0.x, s0.y, s0.z, s1.x, s1.y, s1.z, s0.w, t, u);
  }
};

struct TriLeaf {
  const float4* tri;  // 3 float4 per triangle, original order
  HM_D bool operator()(const BvhView& bvh, const RayInv& r, int leaf, float* t, float* u, int* id) const {
    const int k = __float_as_int(bvh.segs[2 * leaf + 1].w);
    *id = k;
    const float4 a = tri[3 * k], b = tri[3 * k + 1], c = tri[3 * k + 2];
    float v;
    return intersect_triangle(r.ox, r.oy, r.oz, r.dx, r.dy, r.dz, a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, t,
                              u, &v);
  }
};

// Round Catmull-Rom hair: the record holds the segment's box, the control
// points (5 float4 per segment: q0..q3, then strand and end flags) are read
// by id; caps: end caps on (the flags then say which ends have one).
struct CurveLeaf {
  static constexpr int kPrims = 1, kNodes = 2, kChunk = 8;
  const float4* crv;
  int caps;
  HM_D bool operator()(const BvhView& bvh, const RayInv& r, int leaf, float* t, float* u, int* id) const {
    const int k = __float_as_int(bvh.segs[2 * leaf + 1].w);
    *id = k;
    const float4* q = crv + 5 * (size_t)k;
    const int flags = caps ? (int)q[4].y : 0;
    return intersect_curve(r.ox, r.oy, r.oz, r.dx, r.dy, r.dz, q[0], q[1], q[2], q[3], flags, t, u);
  }
};

// Closest hit over the tree's primitives: minimum (t, id) lexicographically.
template <bool kCount>
HM_D void closest_node(const BvhView& bvh, const RayInv& r, TraceStack& st, ClosestState& s, TraceCounters& cnt) {
  if (kCount) cnt.nodes++;
  float t[4];
  int c[4];
  node_boxes(bvh, r, s.cur, s.best_t, t, c);
  // sorting network (Batcher): nearest first, misses (+inf) last
  double e[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) e[k] = hit_key(t[k], c[k]);
  key_swap(e[0], e[1]);
  key_swap(e[2], e[3]);
  key_swap(e[0], e[2]);
  key_swap(e[1], e[3]);
  key_swap(e[1], e[2]);
  if (st.room3()) {
#pragma unroll
    for (int k = 3; k >= 1; --k) st.put(key_child(e[k]), key_hit(e[k]));
    s.cur = key_child(e[0]);
    if (!key_hit(e[0])) s.cur = st.empty() ? kNone : st.pop_lds();
  } else {
#pragma unroll
    for (int k = 3; k >= 1; --k)
      if (key_hit(e[k])) st.push(key_child(e[k]));
    s.cur = key_hit(e[0]) ? key_child(e[0]) : (st.empty() ? kNone : st.pop());
  }
}

template <bool kCount, class Leaf>
HM_D void closest_leaf(const BvhView& bvh, const RayInv& r, TraceStack& st, ClosestState& s, TraceCounters& cnt,
                       const Leaf& leaf_test) {
  const int code = ~s.cur, leaf = code & kLeafPosMask;
  if (kCount) cnt.segs++;
  float t, u;
  int id;
  if (leaf_test(bvh, r, leaf, &t, &u, &id)) {
    if (t < s.best_t || (t == s.best_t && id < s.best_id)) {
      s.best_t = t;
      s.best_id = id;
      s.best_u = u;
    }
  }
  // the rest of a leaf run, one primitive per step
  s.cur = leaf_rest(code);
  if (!s.cur) s.cur = st.empty() ? kNone : st.pop();
}

// A whole query by one lane: the closest hit before (best_t, best_id), or, with
// `first`, the first one found.
template <bool kCount, class Leaf>
HM_D void trace_closest(const BvhView& bvh, const RayInv& r, TraceStack& st, float& best_t, int& best_id,
                        float& best_u, bool first, TraceCounters& cnt, const Leaf& leaf_test) {
  ClosestState s;
  s.best_t = best_t;
  s.best_id = best_id;
  s.best_u = best_u;
  closest_begin(bvh, st, s);
  for (int left = trace_cap(bvh); s.cur != kNone && left > 0; --left) {
    if (s.cur < 0) {
      closest_leaf<kCount, Leaf>(bvh, r, st, s, cnt, leaf_test);
      if (first && s.best_id != best_id) break;
    } else {
      closest_node<kCount>(bvh, r, st, s, cnt);
    }
  }
  best_t = s.best_t;
  best_id = s.best_id;
  best_u = s.best_u;
}

#endif  // __HIPCC__

}  // namespace hm
