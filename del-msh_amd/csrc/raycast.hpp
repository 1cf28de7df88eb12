// raycast.hpp -- per-pixel BVH ray-cast and depth on gfx950.
//
// Semantics are those of del-msh-cpu's recursive first_intersection_ray
// (search_bvh3.rs:103-221) with dis = +inf, not the unordered DFS of the
// reference CUDA kernel:
//   F(node): AABB miss -> none; leaf -> triangle hit with t < inf;
//            both children missed -> none; near = left iff (tl_min, tl_max) <
//            (tr_min, tr_max) lexicographically (else right; a single hit
//            child is near); rn = F(near); if rn and the far entry t > rn.t
//            (or far missed) -> rn; else rf = F(far) and the result is
//            rn if rn.t < rf.t else rf.
// Executed as a flat closest-hit search with the same result: one best hit,
// a stack of 8-byte frames (far child, far entry t) pushed where both children
// are hit (a single hit child is a tail call), a popped far child skipped when
// its entry t exceeds the best t so far, and a triangle hit replacing the best
// when its t <= the best t.  Children are visited near first, so of two hits
// the later one lies in the far subtree of their lowest common ancestor,
// where F's combine keeps far on equal t; a skipped subtree cannot hold a hit
// with t <= the final one.  (The oracle checks this search against the
// recursion on scenes of exact ties: duplicated triangles, rays through grid
// vertices, coplanar soups.)
//
// Layout: before traversal the BVH is packed into
//   inner[i] (64 B, internal node i): both child boxes + both child refs
//   leaf[k]  (48 B, leaf k):          the triangle's three vertices + its id
// so one node expansion is one 64-byte load and one leaf test one 48-byte load
// (the reference layout needs a row load, then dependent box / index / vertex
// gathers).  The values are copies, so the arithmetic is unchanged.
//
// Stack: a lane's last S frames at most sit in LDS ([frame][lane], conflict-free
// for 64-bit accesses), up to kSpillFrames more in its wave's spill area in the
// workspace (SplitStack).  A lane that needs more is searched again alone, with
// the whole spill area of its wave (kDeepFrames frames) as its stack; beyond
// that it raises DMSH_DEVERR_STACK.  So one launch serves every ray, and S can be small
// enough for 26 waves on a CU.  Pixels go to waves in 8x8 tiles; a fixed grid of
// waves takes tiles until none is left (TileDeal).
#pragma once

#include "dmsh_common.hpp"
#include "mat4.hpp"

namespace dmsh {
namespace rc {

constexpr uint32_t kLeafBit = 0x40000000u;   // child ref: leaf slot
constexpr uint32_t kIndexMask = 0x3FFFFFFFu;
constexpr uint32_t kMaxTri = 0x3FFFFFFFu;    // child refs hold 30-bit indices
constexpr int kSpillFrames = 64;                // spilled frames per lane
constexpr uint32_t kDeepFrames = 64u * kSpillFrames;  // a lone lane's frames
constexpr uint32_t kXcds = 8;
constexpr uint32_t kCastCounts = 32 + 32 * kXcds;  // words of CastState::counts

// Bounds of what the regular test serves: boxes and origins within kRegularMax
// and, on one axis, a reciprocal within kRegularInv give a finite t there, as
// 2 * 2^62 * 2^64 = 2^127 is below the largest float.
constexpr float kRegularMax = 0x1p62f, kRegularInv = 0x1p64f;

enum : int { kTraceOk = 0, kTraceOverflow = 1 };

struct alignas(16) InnerNode {
  float4 a;  // c0.lo.xyz, c0.hi.x
  float4 b;  // c0.hi.yz, c1.lo.xy
  float4 c;  // c1.lo.z, c1.hi.xyz
  uint4 d;   // ref c0, ref c1, -, -
};
struct alignas(16) LeafTri {
  float4 a;  // p0.xyz, p1.x
  float4 b;  // p1.yz, p2.xy
  float4 c;  // p2.z, tri id (bits), -, -
};

struct Packed {
  const InnerNode* __restrict__ inner;
  const LeafTri* __restrict__ leaf;
  const float* __restrict__ root_box;  // bvhnode2aabb row 0
  uint32_t num_leaf;
};

// ---------------------------------------------------------------------------
// packing
// ---------------------------------------------------------------------------
// A child id in the LBVH layout: ids from num_leaf - 1 on are leaves.  The
// child's own row is not read here: every row's shape is checked by the
// thread that packs it (an internal row has a second child, a leaf row
// none), which raises DMSH_DEVERR_INDEX and packs a never-hit node or
// triangle for a row that does not fit its place in the layout.
__device__ __forceinline__ uint32_t child_ref(uint32_t c, uint32_t num_leaf, bool& bad) {
  const uint32_t nb = num_leaf - 1, num_node = 2 * num_leaf - 1;
  if (c >= num_node) {
    bad = true;
    return 0;
  }
  return c >= nb ? (kLeafBit | (c - nb)) : c;
}

// The record of an internal node with children (c0, c1) whose boxes are b0,
// b1 (six floats each, read only when the children fit the layout).
template <typename Box6>
__device__ __forceinline__ void store_inner(InnerNode* __restrict__ inner, uint32_t i,
                                            uint32_t c0, uint32_t c1, const Box6& b0,
                                            const Box6& b1, uint32_t num_leaf,
                                            uint32_t* __restrict__ nonfinite,
                                            uint32_t* __restrict__ err) {
  bool bad = (c1 == DMSH_U32MAX);
  const uint32_t r0 = child_ref(c0, num_leaf, bad);
  const uint32_t r1 = child_ref(c1, num_leaf, bad);
  InnerNode nd;
  if (bad) {
    raise_error(err, DMSH_DEVERR_INDEX);
    // an inverted box on both sides: every ray misses this node (in the
    // general slab test, which the flag selects)
    atomicOr(nonfinite, 1u);
    nd.a = make_float4(1.f, 1.f, 1.f, 0.f);
    nd.b = make_float4(0.f, 0.f, 1.f, 1.f);
    nd.c = make_float4(1.f, 0.f, 0.f, 0.f);
    nd.d = make_uint4(kLeafBit, kLeafBit, 0u, 0u);
  } else {
    nd.a = make_float4(b0[0], b0[1], b0[2], b0[3]);
    nd.b = make_float4(b0[4], b0[5], b1[0], b1[1]);
    nd.c = make_float4(b1[2], b1[3], b1[4], b1[5]);
    nd.d = make_uint4(r0, r1, 0u, 0u);
    bool fin = true;
#pragma unroll
    for (int k = 0; k < 6; ++k)
      fin = fin && fabsf(b0[k]) <= kRegularMax && fabsf(b1[k]) <= kRegularMax;
#pragma unroll
    for (int k = 0; k < 3; ++k) fin = fin && b0[k] <= b0[k + 3] && b1[k] <= b1[k + 3];
    if (!fin) atomicOr(nonfinite, 1u);
  }
  inner[i] = nd;
}

// 16-byte part `part` of the record store_inner writes for children (c0,
// c1): parts 0..2 hold the children's bounds x0..x3 (box 0 bounds 0-3;
// bounds 4, 5 of box 0 and 0, 1 of box 1; box 1 bounds 2-5), part 3 the
// refs.  A record whose children do not fit the layout raises (part 0), is
// the one every ray misses and sets *nonfinite, as a part with a bound outside
// +-kRegularMax does (the boxes here are the refit's own: with finite bounds
// lo <= hi).  Writing the four parts from consecutive threads makes a
// wave's store one contiguous kilobyte.
__device__ __forceinline__ uint4 inner_part_bits(uint32_t part, uint32_t c0, uint32_t c1,
                                                 float x0, float x1, float x2, float x3,
                                                 uint32_t num_leaf,
                                                 uint32_t* __restrict__ nonfinite,
                                                 uint32_t* __restrict__ err) {
  bool bad = (c1 == DMSH_U32MAX);
  const uint32_t r0 = child_ref(c0, num_leaf, bad);
  const uint32_t r1 = child_ref(c1, num_leaf, bad);
  if (bad) {
    if (part == 0u) {
      raise_error(err, DMSH_DEVERR_INDEX);
      atomicOr(nonfinite, 1u);
    }
    if (part == 3u) return make_uint4(kLeafBit, kLeafBit, 0u, 0u);
    const float4 e = part == 0u   ? make_float4(1.f, 1.f, 1.f, 0.f)
                     : part == 1u ? make_float4(0.f, 0.f, 1.f, 1.f)
                                  : make_float4(1.f, 0.f, 0.f, 0.f);
    return make_uint4(__float_as_uint(e.x), __float_as_uint(e.y), __float_as_uint(e.z),
                      __float_as_uint(e.w));
  }
  if (part == 3u) return make_uint4(r0, r1, 0u, 0u);
  const bool fin = fabsf(x0) <= kRegularMax && fabsf(x1) <= kRegularMax &&
                   fabsf(x2) <= kRegularMax && fabsf(x3) <= kRegularMax;
  if (!fin) atomicOr(nonfinite, 1u);
  return make_uint4(__float_as_uint(x0), __float_as_uint(x1), __float_as_uint(x2),
                    __float_as_uint(x3));
}

// Internal node i (i + 1 < num_leaf) of one tree into inner[i].
__device__ __forceinline__ void pack_inner(InnerNode* __restrict__ inner,
                                           const uint32_t* __restrict__ bvhnodes,
                                           const float* __restrict__ aabb, uint32_t num_leaf,
                                           uint32_t i, uint32_t* __restrict__ nonfinite,
                                           uint32_t* __restrict__ err) {
  const uint32_t* row = bvhnodes + (size_t)i * 3;
  const uint32_t c0 = row[1], c1 = row[2];
  const uint32_t num_node = 2 * num_leaf - 1;
  // the box pointers are formed only for children inside the tree
  const float* b0 = aabb + (size_t)(c0 < num_node ? c0 : 0u) * 6;
  const float* b1 = aabb + (size_t)(c1 < num_node ? c1 : 0u) * 6;
  store_inner(inner, i, c0, c1, b0, b1, num_leaf, nonfinite, err);
}

// Leaf k of one tree into leaf[k].
__device__ __forceinline__ void pack_leaf(LeafTri* __restrict__ leaf,
                                          const uint32_t* __restrict__ bvhnodes,
                                          const uint32_t* __restrict__ tri2vtx,
                                          const float* __restrict__ xyz, uint32_t num_leaf,
                                          uint32_t num_tri, uint32_t num_vtx, uint32_t k,
                                          uint32_t* __restrict__ err) {
  const uint32_t* row = bvhnodes + (size_t)(num_leaf - 1 + k) * 3;
  const uint32_t tri = row[1];
  LeafTri lt;
  bool ok = row[2] == DMSH_U32MAX && tri < num_tri;
  uint32_t v[3] = {0, 0, 0};
  if (ok) {
    const uint32_t* tv = tri2vtx + (size_t)tri * 3;
    v[0] = tv[0];
    v[1] = tv[1];
    v[2] = tv[2];
    ok = v[0] < num_vtx && v[1] < num_vtx && v[2] < num_vtx;
  }
  if (!ok) {
    raise_error(err, DMSH_DEVERR_INDEX);
    // a degenerate triangle: never hit
    lt.a = make_float4(0.f, 0.f, 0.f, 0.f);
    lt.b = make_float4(0.f, 0.f, 0.f, 0.f);
    lt.c = make_float4(0.f, __uint_as_float(DMSH_U32MAX), 0.f, 0.f);
  } else {
    const float* p0 = xyz + (size_t)v[0] * 3;
    const float* p1 = xyz + (size_t)v[1] * 3;
    const float* p2 = xyz + (size_t)v[2] * 3;
    lt.a = make_float4(p0[0], p0[1], p0[2], p1[0]);
    lt.b = make_float4(p1[1], p1[2], p2[0], p2[1]);
    lt.c = make_float4(p2[2], __uint_as_float(tri), 0.f, 0.f);
  }
  leaf[k] = lt;
}

// The whole tree in one launch: threads [0, num_leaf - 1) pack the internal
// nodes, the next num_leaf the leaves.
static __global__ __launch_bounds__(256) void k_pack_tree(
    InnerNode* __restrict__ inner, LeafTri* __restrict__ leaf,
    const uint32_t* __restrict__ bvhnodes, const float* __restrict__ aabb,
    const uint32_t* __restrict__ tri2vtx, const float* __restrict__ xyz, uint32_t num_leaf,
    uint32_t num_vtx, uint32_t* __restrict__ nonfinite, uint32_t* __restrict__ err) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nb = num_leaf - 1;
  if (i < nb) {
    pack_inner(inner, bvhnodes, aabb, num_leaf, i, nonfinite, err);
  } else if (i - nb < num_leaf) {
    pack_leaf(leaf, bvhnodes, tri2vtx, xyz, num_leaf, num_leaf, num_vtx, i - nb, err);
  }
}

// ---------------------------------------------------------------------------
// traversal
// ---------------------------------------------------------------------------
struct Hit {
  bool has;
  float t;
  uint32_t tri;
};

// A frame: the child ref in the low half, its entry t's bits in the high one.
__device__ __forceinline__ uint64_t make_frame(uint32_t ref, float t) {
  return (uint64_t)__float_as_uint(t) << 32 | ref;
}
__device__ __forceinline__ float frame_t(uint64_t f) { return __uint_as_float((uint32_t)(f >> 32)); }

// LDS words by an LDS pointer: through a generic one the stack's accesses
// become flat memory instructions, which also wait for the vector memory
// (the serving cast took 2.8 instead of 1.5 ms).
using LdsFrame = __attribute__((address_space(3))) uint64_t;

constexpr uint32_t kNoTest = DMSH_U32MAX;

// What is pushed in place of a frame that finds no room: a leaf at t = +inf.
constexpr uint64_t kNoRoom = (uint64_t)0x7F800000u << 32 | kLeafBit;

// A lane's frames: the upper ones, S at most, in LDS, those below them in its
// wave's spill area.  They move half a column at a time, when the LDS column is
// full or empty, so a push or pop in between does not ask where its frame lies:
// with every frame's place decided by its number (below S or not) a step took 6 %
// longer, and perspective casts of 0.3 to 2 million rays were up to 17 % slower
// than with frames in LDS alone.  (104,000 triangles at 1021 x 767: 325 us with
// 20 frames in LDS and restart tiers, 373 then, 339 now.)
// A push that finds the spill column full drops all frames and sets `next`, the
// child that the search would go on with, to kNoTest, which ends it; overflow()
// then says that it counts for nothing.  Neither leaves the loop, which a step
// would pay for too (3 %).  lds and spill point at the lane's column of 64.
template <int S>
struct SplitStack {
  LdsFrame* lds;
  uint64_t* spill;
  int sp = 0;     // frames in LDS
  int below = 0;  // frames in the spill area
  bool full = false;
  static constexpr int kHalf = S / 2;
  __device__ __forceinline__ void push(uint64_t f, uint32_t& next) {
    if (__builtin_expect(sp == S, 0)) {
      if (below + kHalf > kSpillFrames) {
        full = true;
        sp = below = 0;
        next = kNoTest;
        f = kNoRoom;
      } else {
#pragma unroll
        for (int k = 0; k < kHalf; ++k) spill[(below + k) * 64] = lds[k * 64];
#pragma unroll
        for (int k = kHalf; k < S; ++k) lds[(k - kHalf) * 64] = lds[k * 64];
        below += kHalf;
        sp -= kHalf;
      }
    }
    lds[sp * 64] = f;
    ++sp;
  }
  // Pops to the next frame whose entry t does not exceed `best`; false when
  // none is left.
  __device__ __forceinline__ bool pop(float best, uint64_t& f) {
    for (;;) {
      while (sp > 0) {
        --sp;
        f = lds[sp * 64];
        if (!(frame_t(f) > best)) return true;
      }
      if (below == 0) return false;
      below -= kHalf;
#pragma unroll
      for (int k = 0; k < kHalf; ++k) lds[k * 64] = spill[(below + k) * 64];
      sp = kHalf;
    }
  }
  __device__ __forceinline__ bool overflow() const { return full; }
};

// One lane's frames in a run of kDeepFrames words of global memory.
struct DeepStack {
  uint64_t* base;
  uint32_t sp = 0;
  bool full = false;
  __device__ __forceinline__ void push(uint64_t f, uint32_t& next) {
    if (sp == kDeepFrames) {
      full = true;
      sp = 0;
      next = kNoTest;
      f = kNoRoom;
    }
    base[sp++] = f;
  }
  __device__ __forceinline__ bool pop(float best, uint64_t& f) {
    while (sp > 0) {
      f = base[--sp];
      if (!(frame_t(f) > best)) return true;
    }
    return false;
  }
  __device__ __forceinline__ bool overflow() const { return full; }
};

// Rust's tuple `<` on (tmin, tmax).
__device__ __forceinline__ bool tuple_lt(float a0, float a1, float b0, float b1) {
  return (a0 == b0) ? (a1 < b1) : (a0 < b0);
}

__device__ __forceinline__ void leaf_test(const Packed& pk, uint32_t slot, const float org[3],
                                          const float dir[3], bool& has, float& t_out,
                                          uint32_t& tri_out) {
  const LeafTri lt = pk.leaf[slot];
  const float p0[3] = {lt.a.x, lt.a.y, lt.a.z};
  const float p1[3] = {lt.a.w, lt.b.x, lt.b.y};
  const float p2[3] = {lt.b.z, lt.b.w, lt.c.x};
  float t;
  has = tri_intersect(p0, p1, p2, org, dir, true, t, nullptr) && (t < __builtin_inff());
  t_out = has ? t : 0.f;
  tri_out = has ? __float_as_uint(lt.c.y) : DMSH_U32MAX;
}

// Slab test for a regular ray (see regular_ray) against a box within
// +-kRegularMax with lo <= hi.  The plane a ray enters through is lo for a
// positive reciprocal and hi for a negative one: with lo <= hi and correctly
// rounded (so monotone) subtraction and product that t is the smaller of the
// two, so selecting the plane gives what the general test's compare-and-select
// gives, up to the sign of a zero, which no later comparison can see.  A
// parallel axis carries the
// reciprocal +inf: lo < o gives -inf, lo > o gives +inf, and lo == o gives NaN,
// which fmaxf ignores as it would -inf (for hi: fminf, +inf); so an origin
// inside the slab leaves the axis out, as the general test does, and one
// outside leaves tmax = -inf, or tmin = +inf with the finite tmax of the axis
// whose t cannot overflow (regular_ray sees to one), and misses.
__device__ __forceinline__ bool slab_hit_regular(const RaySlab& r, const bool neg[3],
                                                 const float lo[3], const float hi[3],
                                                 float& tmin_out, float& tmax_out) {
  float tn[3], tf[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    tn[i] = ((neg[i] ? hi[i] : lo[i]) - r.o[i]) * r.inv[i];
    tf[i] = ((neg[i] ? lo[i] : hi[i]) - r.o[i]) * r.inv[i];
  }
  const float tmin = fmaxf(fmaxf(tn[0], tn[1]), tn[2]);
  const float tmax = fminf(fminf(tf[0], tf[1]), tf[2]);
  tmin_out = tmin;
  tmax_out = tmax;
  return !(tmin > tmax) && !(tmax < 0.f);
}

// Whether slab_hit_regular serves this ray: an origin within the bound, per axis
// a nonzero reciprocal that is finite or of a parallel axis, and one of them
// within its bound.  Makes the reciprocals of parallel axes +inf.
__device__ __forceinline__ bool regular_ray(RaySlab& r, bool neg[3]) {
  bool ok = true, some = false;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float a = fabsf(r.inv[i]);
    ok = ok && a > 0.f && fabsf(r.o[i]) <= kRegularMax;  // false for a NaN
    some = some || a <= kRegularInv;
  }
  ok = ok && some;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (ok && r.par[i]) r.inv[i] = __builtin_inff();
    neg[i] = r.inv[i] < 0.f;
  }
  return ok;
}

// The traversal loop.  An iteration first pops, if the lane has no node to
// expand, the next far child not skipped by the best hit (ending the lane's
// search when the stack runs out); then expands the lane's node, if any; then
// runs the (single) leaf-test site if the pop or the expansion produced a
// leaf, so a wave whose lanes diverge between these steps pays for the
// triangle test once.  best is +inf until a triangle is hit.
template <bool kRegular, class Stack>
__device__ __forceinline__ int trace_loop(const Packed& pk, const RaySlab& r, const bool neg[3],
                                          const float org[3], const float dir[3], Stack& stk,
                                          Hit& out) {
  float best = __builtin_inff();
  uint32_t best_tri = DMSH_U32MAX;
  uint32_t node = 0;
  bool expand = true;
  for (;;) {
    uint32_t test = kNoTest;
    if (!expand) {
      uint64_t f;
      if (!stk.pop(best, f)) break;
      node = (uint32_t)f;
      expand = !(node & kLeafBit);
      if (!expand) test = node & kIndexMask;
    }
    if (expand) {
      const InnerNode nd = pk.inner[node];
      const float l0[3] = {nd.a.x, nd.a.y, nd.a.z}, h0[3] = {nd.a.w, nd.b.x, nd.b.y};
      const float l1[3] = {nd.b.z, nd.b.w, nd.c.x}, h1[3] = {nd.c.y, nd.c.z, nd.c.w};
      float tl0, tl1, tr0, tr1;
      bool hl, hr;
      if (kRegular) {
        hl = slab_hit_regular(r, neg, l0, h0, tl0, tl1);
        hr = slab_hit_regular(r, neg, l1, h1, tr0, tr1);
      } else {
        hl = slab_hit(r, l0, h0, tl0, tl1);
        hr = slab_hit(r, l1, h1, tr0, tr1);
      }
      uint32_t next = kNoTest;
      if (hl && hr) {
        const bool nl = tuple_lt(tl0, tl1, tr0, tr1);
        const float tfar = nl ? tr0 : tl0;
        next = nl ? nd.d.x : nd.d.y;
        // a far child beyond the best hit would only be skipped later
        if (!(tfar > best)) stk.push(make_frame(nl ? nd.d.y : nd.d.x, tfar), next);
      } else if (hl || hr) {
        next = hl ? nd.d.x : nd.d.y;
      }
      if (next == kNoTest) {
        expand = false;  // both children missed
      } else if (next & kLeafBit) {
        test = next & kIndexMask;
        expand = false;
      } else {
        node = next;
      }
    }
    if (test != kNoTest) {
      bool has;
      float t;
      uint32_t tri;
      leaf_test(pk, test, org, dir, has, t, tri);
      if (has && t <= best) {
        best = t;
        best_tri = tri;
      }
    }
  }
  out.has = best < __builtin_inff();
  out.t = best;
  out.tri = best_tri;
  return stk.overflow() ? kTraceOverflow : kTraceOk;
}

// regular: every packed child box lies within +-kRegularMax with lo <= hi
// (checked while packing).
template <class Stack>
__device__ __forceinline__ int trace(const Packed& pk, const float org[3], const float dir[3],
                                     Stack& stk, Hit& out, bool regular) {
  out.has = false;
  out.t = 0.f;
  out.tri = DMSH_U32MAX;
  if (pk.num_leaf == 0) return kTraceOk;
  RaySlab r;
  make_slab(org, dir, r);
  {
    const float lo[3] = {pk.root_box[0], pk.root_box[1], pk.root_box[2]};
    const float hi[3] = {pk.root_box[3], pk.root_box[4], pk.root_box[5]};
    float ta, tb;
    if (!slab_hit(r, lo, hi, ta, tb)) return kTraceOk;
  }
  if (pk.num_leaf == 1) {
    leaf_test(pk, 0, org, dir, out.has, out.t, out.tri);
    return kTraceOk;
  }
  // one path for all lanes still here
  bool neg[3];
  RaySlab q = r;
  if (__all(regular && regular_ray(q, neg)))
    return trace_loop<true>(pk, q, neg, org, dir, stk, out);
  return trace_loop<false>(pk, r, neg, org, dir, stk, out);
}

// Tiles of the images of one launch, dealt to a fixed grid of waves.  Chunks
// of neighbouring tiles go to the XCDs in turn: their rays share BVH nodes in
// one L2, and every XCD gets a like share of the work, so no wave has to look
// for tiles elsewhere.  A wave's first tile is that of its own place in its
// XCD's list, the later ones come from the XCD's ticket counter one at a time.
// (Device-scope atomics on one word run ~14 ns one after another: when every
// wave also went past the other XCDs' counters at the end, that alone took 60 us
// of a launch.  Runs of 2 to 8 tiles a ticket, or a fixed share with tickets
// only for the rest, were slower: 24 requests of 7.3 M rays in all 1.61 ms with
// single tiles, 1.78 with runs of 2, 1.86 with 8, 1.79 to 2.0 with a fixed
// share.)
struct TileDeal {
  uint32_t* ticket;        // of this XCD
  uint32_t shift;          // log2 of the chunk
  uint32_t groups, group;  // XCDs in use, this wave's
  uint32_t len;            // tiles (some past the end) of this XCD
  uint32_t waves;          // waves of this XCD
  uint32_t own;            // this wave's first, then kTaken
  static constexpr uint32_t kTaken = DMSH_U32MAX;

  template <int W>
  static __device__ __forceinline__ TileDeal make(uint32_t* counts, uint32_t num_tiles) {
    TileDeal d;
    d.groups = gridDim.x < kXcds ? gridDim.x : kXcds;
    d.group = blockIdx.x % d.groups;
    d.ticket = counts + 32u + 32u * d.group;
    // chunks of up to 256 tiles, at least 16 of them on each XCD
    const uint32_t want = num_tiles / (d.groups * 16u);
    d.shift = want == 0u ? 0u : 31u - (uint32_t)__builtin_clz(want);
    if (d.shift > 8u) d.shift = 8u;
    const uint32_t round = d.groups << d.shift;
    d.len = (num_tiles / round + (num_tiles % round != 0u ? 1u : 0u)) << d.shift;
    d.waves = (gridDim.x + d.groups - 1u - d.group) / d.groups * (uint32_t)W;
    d.own = blockIdx.x / d.groups * (uint32_t)W + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    return d;
  }
  // the next tile, the same in every lane (it may be past the end); false
  // when none is left
  __device__ __forceinline__ bool next(uint32_t& tile) {
    uint32_t q = own;
    if (q == kTaken) {
      if (waves >= len) return false;
      uint32_t t = 0u;
      if ((threadIdx.x & 63u) == 0u) t = atomicAdd(ticket, 1u);
      q = waves + __builtin_amdgcn_readfirstlane(t);
    }
    own = kTaken;
    if (q >= len) return false;
    tile = (((q >> shift) * groups + group) << shift) + (q & ((1u << shift) - 1u));
    return true;
  }
};

// Largest m < M with off[m] <= x (off[0] <= x; off ascending), by the whole
// wave: 64 entries a round trip.
__device__ __forceinline__ uint32_t wave_segment(const uint32_t* __restrict__ off, uint32_t M,
                                                 uint32_t x) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t lo = 0u, n = M;
  for (;;) {
    const uint32_t step = n / 64u + (n % 64u != 0u ? 1u : 0u);
    const bool mine = lane * step < n;
    const uint64_t below = __ballot(mine && off[lo + (mine ? lane * step : 0u)] <= x);
    const uint32_t k = ((uint32_t)__popcll(below) - 1u) * step;
    lo += k;
    if (step == 1u) return lo;
    n = n - k < step ? n - k : step;
  }
}

// Upper bound of the 8x8 tiles of `images` images with num_pix pixels in all:
// a w x h image has at most (w / 8 + 1)(h / 8 + 1) <= wh (1/64 + 1/8) + 9/8.
inline uint32_t max_tiles(uint64_t num_pix, uint64_t images) {
  const uint64_t t = num_pix * 9u / 64u + 2u * images + 1u;
  return t < num_pix ? (uint32_t)t : (uint32_t)num_pix;
}
// Waves per CU in workgroups of W that fit its 160 KB of LDS with S frames a
// lane (of the 32 waves that their registers allow).  A grid of more would start
// the last workgroups when others have ended, and those with their own first
// tiles.
constexpr uint32_t resident_waves(int S, int W) {
  const uint32_t by_lds = 160u * 1024u / (uint32_t)(S * 512 * W), by_regs = 32u / (uint32_t)W;
  return (by_lds < by_regs ? by_lds : by_regs) * (uint32_t)W;
}
static_assert(resident_waves(12, 1) == 26 && resident_waves(12, 2) == 26 &&
                  resident_waves(12, 4) == 24 && resident_waves(32, 4) == 8,
              "whole workgroups");
// Waves of a launch over at most `tiles` tiles with any number of frames, and
// the words of spill area each of them owns: 32 KB, so 208 MiB from 6656 tiles
// (a 649 x 649 image) on.
constexpr int kMinFrames = 12;
constexpr uint32_t kMaxCastWaves = 256u * resident_waves(kMinFrames, 1);
inline uint32_t cast_waves(uint32_t tiles) { return tiles < kMaxCastWaves ? tiles : kMaxCastWaves; }
constexpr size_t kSpillPerWave = (size_t)kSpillFrames * 64;

struct CastState {
  uint32_t* counts;  // [kCastCounts]: [2] nonzero when a box is not regular (one
                     // tree, batch), [3] offsets rejected, [32 + 32 x] tickets of XCD x: each on
                     // a 128-byte line of its own, away from the flags, which
                     // every tile reads (a load waits behind the line's atomics)
  uint64_t* spill;   // [waves][kSpillPerWave]
  uint32_t* err;
};

// One wave's share of a launch.  Src: num_tiles(), and load(tile, lane, job)
// for the pixel of a lane: whether it lies in its image, its ray's transform
// (16 floats, column-major), tree and output position.
struct PixelJob {
  Packed pk;
  const float* T;
  uint32_t iw, ih, w, h;
  uint32_t out;
  bool regular;
};

template <int S, int W, class Src>
__device__ __forceinline__ void cast_wave(const Src& src, const CastState& st, LdsFrame* lds,
                                          uint32_t* __restrict__ pix2tri,
                                          float* __restrict__ pix2t) {
  const uint32_t lane = threadIdx.x & 63u;
  uint64_t* spill = st.spill + (size_t)(blockIdx.x * (uint32_t)W +
                                     __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) *
                                kSpillPerWave;
  const uint32_t num_tiles = src.num_tiles();
  TileDeal deal = TileDeal::make<W>(st.counts, num_tiles);
  uint32_t tile;
  while (deal.next(tile)) {
    if (tile >= num_tiles) continue;
    PixelJob j;
    const bool in = src.load(tile, lane, j);
    bool deep = false;
    float org[3], dir[3];
    Hit hit;
    if (in) {
      float m[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) m[k] = j.T[k];
      ray_for_pixel(j.iw, j.ih, j.w, j.h, m, org, dir);
      SplitStack<S> stk{lds + lane, spill + lane};
      deep = trace(j.pk, org, dir, stk, hit, j.regular) == kTraceOverflow;
    }
    // lanes that ran out of frames, one after the other
    for (uint64_t left = __ballot(deep); left != 0; left &= left - 1) {
      if (lane == (uint32_t)__builtin_ctzll(left)) {
        DeepStack stk{spill};
        if (trace(j.pk, org, dir, stk, hit, false) != kTraceOk) {
          raise_error(st.err, DMSH_DEVERR_STACK);
          hit.has = false;
        }
      }
    }
    if (in) {
      pix2tri[j.out] = hit.has ? hit.tri : DMSH_U32MAX;
      if (pix2t) pix2t[j.out] = hit.has ? hit.t : 0.f;
    }
  }
}

// A single image of one tree.
struct ImageSrc {
  Packed pk;
  const float* T;
  uint32_t img_w, img_h, tiles_x, tiles;
  const uint32_t* counts;
  __device__ __forceinline__ uint32_t num_tiles() const { return tiles; }
  __device__ __forceinline__ bool load(uint32_t tile, uint32_t lane, PixelJob& j) const {
    j.pk = pk;
    j.T = T;
    j.w = img_w;
    j.h = img_h;
    j.iw = (tile % tiles_x) * 8u + (lane & 7u);
    j.ih = (tile / tiles_x) * 8u + (lane >> 3);
    j.out = j.ih * img_w + j.iw;
    j.regular = counts[2] == 0u;
    return j.iw < img_w && j.ih < img_h;
  }
};

template <int S, int W>
__global__ __launch_bounds__(64 * W) void k_pix2tri(ImageSrc src, CastState st,
                                                    uint32_t* __restrict__ pix2tri,
                                                    float* __restrict__ pix2t) {
  __shared__ uint64_t s_stack[W][S][64];
  cast_wave<S, W>(src, st, (LdsFrame*)&s_stack[threadIdx.x >> 6][0][0], pix2tri, pix2t);
}

__device__ __forceinline__ void load_transform(const float* __restrict__ T, float m[16]) {
#pragma unroll
  for (int k = 0; k < 16; ++k) m[k] = T[k];
}

// ---------------------------------------------------------------------------
// depth
// ---------------------------------------------------------------------------

struct TriMesh {
  const uint32_t* __restrict__ tri2vtx;
  const float* __restrict__ xyz;
  uint32_t num_tri, num_vtx;
};

static __global__ __launch_bounds__(256) void k_pix2depth(float* __restrict__ depth,
                                                          const uint32_t* __restrict__ pix2tri,
                                                          TriMesh sc, uint32_t img_w,
                                                          uint32_t img_h,
                                                          const float* __restrict__ T,
                                                          const float* __restrict__ inv,
                                                          uint32_t* __restrict__ err) {
  const uint32_t ip = blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= img_w * img_h) return;
  const uint32_t tri = pix2tri[ip];
  float out = 0.f;
  if (tri != DMSH_U32MAX && inv[16] != 0.f) {
    if (tri >= sc.num_tri) {
      raise_error(err, DMSH_DEVERR_INDEX);
    } else {
      const uint32_t* tv = sc.tri2vtx + (size_t)tri * 3;
      const uint32_t i0 = tv[0], i1 = tv[1], i2 = tv[2];
      if (i0 >= sc.num_vtx || i1 >= sc.num_vtx || i2 >= sc.num_vtx) {
        raise_error(err, DMSH_DEVERR_INDEX);
      } else {
        float m[16], w2n[16];
        load_transform(T, m);
        load_transform(inv, w2n);
        const uint32_t ih = ip / img_w, iw = ip - ih * img_w;
        float org[3], dir[3], p0[3], p1[3], p2[3], t;
        ray_for_pixel(iw, ih, img_w, img_h, m, org, dir);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          p0[k] = sc.xyz[(size_t)i0 * 3 + k];
          p1[k] = sc.xyz[(size_t)i1 * 3 + k];
          p2[k] = sc.xyz[(size_t)i2 * 3 + k];
        }
        if (tri_intersect(p0, p1, p2, org, dir, false, t, nullptr)) {
          const float pos[3] = {t * dir[0] + org[0], t * dir[1] + org[1], t * dir[2] + org[2]};
          float ndc[3];
          if (transform_homogeneous(w2n, pos[0], pos[1], pos[2], ndc)) out = (ndc[2] + 1.f) * 0.5f;
        }
      }
    }
  }
  depth[ip] = out;
}

// d transform_homogeneous(m, p) / d p, rows 0..2 (quotient rule):
// J[r][j] = (m[j*4+r] w - x_r m[j*4+3]) / w^2, x_r the numerator of row r.
__device__ __forceinline__ void jacobian_transform3(const float* m, const float p[3],
                                                    float J[3][3]) {
  const float x = p[0], y = p[1], z = p[2];
  const float w = ((m[3] * x + m[7] * y) + m[11] * z) + m[15];
  const float inv_w2 = 1.f / (w * w);
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const float q = ((m[r] * x + m[4 + r] * y) + m[8 + r] * z) + m[12 + r];
#pragma unroll
    for (int j = 0; j < 3; ++j) J[r][j] = (m[j * 4 + r] * w - q * m[j * 4 + 3]) * inv_w2;
  }
}

// Depth backward, one thread per pixel: the line hit (t, bc) of the stored
// triangle, q = sum bc_k p_k, dL/dq = J(world2ndc, q)^T (0, 0, g/2),
// dL/dt = dir . dL/dq, and the hit's sensitivity to the triangle,
// dL/dp_k = (dL/dt / (n . dir)) bc_k n with n = (p1 - p0) x (p2 - p0);
// nine float atomics per covered pixel.
static __global__ __launch_bounds__(256) void k_pix2depth_bwd(
    float* __restrict__ dldw_xyz, const uint32_t* __restrict__ pix2tri, TriMesh sc,
    const float* __restrict__ dldw_depth, uint32_t img_w, uint32_t img_h,
    const float* __restrict__ T, const float* __restrict__ inv, uint32_t* __restrict__ err) {
  const uint32_t ip = blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= img_w * img_h) return;
  const uint32_t tri = pix2tri[ip];
  if (tri == DMSH_U32MAX || inv[16] == 0.f) return;
  if (tri >= sc.num_tri) {
    raise_error(err, DMSH_DEVERR_INDEX);
    return;
  }
  const uint32_t* tv = sc.tri2vtx + (size_t)tri * 3;
  const uint32_t iv[3] = {tv[0], tv[1], tv[2]};
  if (iv[0] >= sc.num_vtx || iv[1] >= sc.num_vtx || iv[2] >= sc.num_vtx) {
    raise_error(err, DMSH_DEVERR_INDEX);
    return;
  }
  float m[16], w2n[16];
  load_transform(T, m);
  load_transform(inv, w2n);
  const uint32_t ih = ip / img_w, iw = ip - ih * img_w;
  float org[3], dir[3], p0[3], p1[3], p2[3], t, bc[3];
  ray_for_pixel(iw, ih, img_w, img_h, m, org, dir);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    p0[k] = sc.xyz[(size_t)iv[0] * 3 + k];
    p1[k] = sc.xyz[(size_t)iv[1] * 3 + k];
    p2[k] = sc.xyz[(size_t)iv[2] * 3 + k];
  }
  if (!tri_intersect(p0, p1, p2, org, dir, false, t, bc)) return;
  float q[3], J[3][3], dldq[3], e1[3], e2[3], n[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) q[i] = (bc[0] * p0[i] + bc[1] * p1[i]) + bc[2] * p2[i];
  jacobian_transform3(w2n, q, J);
  const float half_g = 0.5f * dldw_depth[ip];
#pragma unroll
  for (int j = 0; j < 3; ++j) dldq[j] = (J[0][j] * 0.f + J[1][j] * 0.f) + J[2][j] * half_g;
  const float dldt = dot3(dir, dldq);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    e1[i] = p1[i] - p0[i];
    e2[i] = p2[i] - p0[i];
  }
  cross3(e1, e2, n);
  const float s = dldt / dot3(n, dir);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float sk = s * bc[k];
#pragma unroll
    for (int i = 0; i < 3; ++i) unsafeAtomicAdd(dldw_xyz + (size_t)iv[k] * 3 + i, sk * n[i]);
  }
}

// ---------------------------------------------------------------------------
// attribute interpolation (pix2tri.rs:176-304)
// ---------------------------------------------------------------------------
// Barycentric coordinates of the line (org, dir) against the plane of the
// triangle: Moller-Trumbore's u, v with no range or epsilon test; also the
// reciprocal determinant and the two cross products the backward reuses.
__device__ __forceinline__ void plane_line_bc(const float p0[3], const float p1[3],
                                              const float p2[3], const float org[3],
                                              const float dir[3], float& u, float& v,
                                              float& inv_det, float pvec[3], float e1xd[3]) {
  float e1[3], e2[3], tvec[3], qvec[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    e1[i] = p1[i] - p0[i];
    e2[i] = p2[i] - p0[i];
    tvec[i] = org[i] - p0[i];
  }
  cross3(dir, e2, pvec);
  const float det = dot3(e1, pvec);
  inv_det = 1.f / det;
  u = inv_det * dot3(tvec, pvec);
  cross3(tvec, e1, qvec);
  v = inv_det * dot3(dir, qvec);
  cross3(e1, dir, e1xd);
}

// One thread per pixel: pix2val = bc0 val[i0] + bc1 val[i1] + bc2 val[i2] on
// covered pixels, 0 on the background.
static __global__ __launch_bounds__(256) void k_interpolate(
    float* __restrict__ pix2val, const uint32_t* __restrict__ pix2tri, TriMesh sc,
    uint32_t num_vdim, const float* __restrict__ vtx2val, uint32_t img_w, uint32_t img_h,
    const float* __restrict__ T, uint32_t* __restrict__ err) {
  const uint32_t ip = blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= img_w * img_h) return;
  float* out = pix2val + (size_t)ip * num_vdim;
  const uint32_t tri = pix2tri[ip];
  uint32_t iv[3] = {0u, 0u, 0u};
  bool ok = tri != DMSH_U32MAX;
  if (ok && tri >= sc.num_tri) {
    raise_error(err, DMSH_DEVERR_INDEX);
    ok = false;
  }
  if (ok) {
    const uint32_t* tv = sc.tri2vtx + (size_t)tri * 3;
    iv[0] = tv[0];
    iv[1] = tv[1];
    iv[2] = tv[2];
    if (iv[0] >= sc.num_vtx || iv[1] >= sc.num_vtx || iv[2] >= sc.num_vtx) {
      raise_error(err, DMSH_DEVERR_INDEX);
      ok = false;
    }
  }
  if (!ok) {
    for (uint32_t d = 0; d < num_vdim; ++d) out[d] = 0.f;
    return;
  }
  float m[16];
  load_transform(T, m);
  const uint32_t ih = ip / img_w, iw = ip - ih * img_w;
  float org[3], dir[3], p[3][3], u, v, inv_det, pvec[3], c[3];
  ray_for_pixel(iw, ih, img_w, img_h, m, org, dir);
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int i = 0; i < 3; ++i) p[k][i] = sc.xyz[(size_t)iv[k] * 3 + i];
  plane_line_bc(p[0], p[1], p[2], org, dir, u, v, inv_det, pvec, c);
  const float bc0 = 1.f - u - v;
  for (uint32_t d = 0; d < num_vdim; ++d)
    out[d] = (bc0 * vtx2val[(size_t)iv[0] * num_vdim + d] +
              u * vtx2val[(size_t)iv[1] * num_vdim + d]) +
             v * vtx2val[(size_t)iv[2] * num_vdim + d];
}

// Backward, one thread per covered pixel.  With gu = dL/dbc1 - dL/dbc0 and
// gv = dL/dbc2 - dL/dbc0 (dL/dt = 0), implicit differentiation of
// u e1 + v e2 - t dir = org - p0 gives dL/dp0 = -bc0 lam, dL/dp1 = -u lam,
// dL/dp2 = -v lam with lam = (gu (dir x e2) + gv (e1 x dir)) / det; and
// dL/dval[ik] = dL/dpix bc_k.  Float atomics accumulate both.
static __global__ __launch_bounds__(256) void k_interpolate_bwd(
    float* __restrict__ dldw_xyz, float* __restrict__ dldw_val,
    const uint32_t* __restrict__ pix2tri, TriMesh sc, uint32_t num_vdim,
    const float* __restrict__ vtx2val, const float* __restrict__ dldw_pix2val, uint32_t img_w,
    uint32_t img_h, const float* __restrict__ T, uint32_t* __restrict__ err) {
  const uint32_t ip = blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= img_w * img_h) return;
  const uint32_t tri = pix2tri[ip];
  if (tri == DMSH_U32MAX) return;
  if (tri >= sc.num_tri) {
    raise_error(err, DMSH_DEVERR_INDEX);
    return;
  }
  const uint32_t* tv = sc.tri2vtx + (size_t)tri * 3;
  const uint32_t iv[3] = {tv[0], tv[1], tv[2]};
  if (iv[0] >= sc.num_vtx || iv[1] >= sc.num_vtx || iv[2] >= sc.num_vtx) {
    raise_error(err, DMSH_DEVERR_INDEX);
    return;
  }
  const float* g = dldw_pix2val + (size_t)ip * num_vdim;
  float gb[3] = {0.f, 0.f, 0.f};
  for (uint32_t d = 0; d < num_vdim; ++d) {
    const float gd = g[d];
#pragma unroll
    for (int k = 0; k < 3; ++k) gb[k] += vtx2val[(size_t)iv[k] * num_vdim + d] * gd;
  }
  const float gu = gb[1] - gb[0], gv = gb[2] - gb[0];
  float m[16];
  load_transform(T, m);
  const uint32_t ih = ip / img_w, iw = ip - ih * img_w;
  float org[3], dir[3], p[3][3], u, v, inv_det, pvec[3], c[3];
  ray_for_pixel(iw, ih, img_w, img_h, m, org, dir);
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int i = 0; i < 3; ++i) p[k][i] = sc.xyz[(size_t)iv[k] * 3 + i];
  plane_line_bc(p[0], p[1], p[2], org, dir, u, v, inv_det, pvec, c);
  const float bc[3] = {1.f - u - v, u, v};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float lam = (gu * pvec[i] + gv * c[i]) * inv_det;
#pragma unroll
    for (int k = 0; k < 3; ++k) unsafeAtomicAdd(dldw_xyz + (size_t)iv[k] * 3 + i, -(bc[k] * lam));
  }
  for (uint32_t d = 0; d < num_vdim; ++d) {
    const float gd = g[d];
#pragma unroll
    for (int k = 0; k < 3; ++k) unsafeAtomicAdd(dldw_val + (size_t)iv[k] * num_vdim + d, gd * bc[k]);
  }
}

}  // namespace rc
}  // namespace dmsh
