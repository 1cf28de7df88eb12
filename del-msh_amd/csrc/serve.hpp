// serve.hpp -- kernels behind the serving loop: trees packed into
// self-contained device buffers (one per cached mesh) and one ray-cast
// launch over the images of many requests, each naming its tree by address.
//
// Packed tree of N triangles (dmsh_packed_bytes): inner nodes [N-1] (64 B),
// leaves [N] (48 B), the root box (6 floats), then a word that is nonzero
// when a box of the tree needs the general slab test (rc::store_inner) -- the
// traversal layout of raycast.hpp, so a cast reads nothing else.
#pragma once

#include "batch.hpp"

namespace dmsh {
namespace srv {

struct PackedRef {
  rc::InnerNode* inner;
  rc::LeafTri* leaf;
  float* root_box;
};

__host__ __device__ __forceinline__ size_t packed_leaf_offset(uint32_t n) {
  return (size_t)(n > 1 ? n - 1 : 0) * sizeof(rc::InnerNode);
}
__host__ __device__ __forceinline__ size_t packed_box_offset(uint32_t n) {
  return packed_leaf_offset(n) + (size_t)n * sizeof(rc::LeafTri);
}
__host__ __device__ __forceinline__ size_t packed_flag_offset(uint32_t n) {
  return packed_box_offset(n) + 6 * sizeof(float);
}
__host__ __device__ __forceinline__ size_t packed_bytes(uint32_t n) {
  return packed_flag_offset(n) + sizeof(uint32_t);
}

__device__ __forceinline__ PackedRef packed_ref(uint64_t addr, uint32_t n) {
  char* base = reinterpret_cast<char*>(addr);
  return PackedRef{reinterpret_cast<rc::InnerNode*>(base),
                   reinterpret_cast<rc::LeafTri*>(base + packed_leaf_offset(n)),
                   reinterpret_cast<float*>(base + packed_box_offset(n))};
}
__device__ __forceinline__ uint32_t* packed_flag(uint64_t addr, uint32_t n) {
  return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(addr) + packed_flag_offset(n));
}

// The pack sink of one mesh for the batched refit: its records go straight
// into the mesh's packed buffer, as k_pack_to_buffers writes them.
struct TreePack {
  static constexpr bool kOn = true;
  rc::InnerNode* inner;
  rc::LeafTri* leaf;
  uint32_t* nonfinite;
  // the records rc::pack_leaf writes, from the corners the refit loaded
  __device__ __forceinline__ void leaf_ok(uint32_t k, const float (&p0)[3], const float (&p1)[3],
                                          const float (&p2)[3], uint32_t tri) const {
    rc::LeafTri lt;
    lt.a = make_float4(p0[0], p0[1], p0[2], p1[0]);
    lt.b = make_float4(p1[1], p1[2], p2[0], p2[1]);
    lt.c = make_float4(p2[2], __uint_as_float(tri), 0.f, 0.f);
    leaf[k] = lt;
  }
  __device__ __forceinline__ void leaf_bad(uint32_t k) const {
    rc::LeafTri lt;
    lt.a = make_float4(0.f, 0.f, 0.f, 0.f);
    lt.b = make_float4(0.f, 0.f, 0.f, 0.f);
    lt.c = make_float4(0.f, __uint_as_float(DMSH_U32MAX), 0.f, 0.f);
    leaf[k] = lt;
  }
  // 16-byte part `part` of internal node i's record (rc::inner_part_bits)
  __device__ __forceinline__ void inner_part(uint32_t i, uint32_t part, uint32_t c0, uint32_t c1,
                                             float x0, float x1, float x2, float x3,
                                             uint32_t num_leaf, uint32_t* err) const {
    reinterpret_cast<uint4*>(inner + i)[part] =
        rc::inner_part_bits(part, c0, c1, x0, x1, x2, x3, num_leaf, nonfinite, err);
  }
  __device__ __forceinline__ void inner_at(uint32_t i, uint32_t c0, uint32_t c1,
                                           const float (&b0)[6], const float (&b1)[6],
                                           uint32_t num_leaf, uint32_t* err) const {
    rc::store_inner(inner, i, c0, c1, b0, b1, num_leaf, nonfinite, err);
  }
};

struct PackSrc {
  using PK = TreePack;
  const uint64_t* dst;  // [M] packed buffer addresses
  uint32_t* nonfinite;  // [M], zeroed before the build
  __device__ __forceinline__ TreePack of(uint32_t m, uint32_t n) const {
    const PackedRef p = packed_ref(dst[m], n);
    return TreePack{p.inner, p.leaf, nonfinite + m};
  }
};

// After a build that packed as it refit: each mesh's root box and its
// slab-test flag into its packed buffer.
static __global__ __launch_bounds__(256) void k_pack_roots(uint32_t M,
                                                           const uint32_t* __restrict__ mesh2tri,
                                                           const uint32_t* __restrict__ node_off,
                                                           const float* __restrict__ aabb,
                                                           const uint64_t* __restrict__ dst,
                                                           const uint32_t* __restrict__ nonfinite,
                                                           const uint32_t* __restrict__ bad) {
  const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
  if (*bad || m >= M) return;
  const uint32_t n = mesh2tri[m + 1] - mesh2tri[m];
  if (n == 0) return;
  const PackedRef p = packed_ref(dst[m], n);
#pragma unroll
  for (int d = 0; d < 6; ++d) p.root_box[d] = aabb[(size_t)node_off[m] * 6 + d];
  *packed_flag(dst[m], n) = nonfinite[m];
}

// The per-mesh slab-test flags into the packed buffers (after the pack).
static __global__ __launch_bounds__(256) void k_pack_flags(uint32_t M,
                                                           const uint32_t* __restrict__ mesh2tri,
                                                           const uint64_t* __restrict__ dst,
                                                           const uint32_t* __restrict__ nonfinite,
                                                           const uint32_t* __restrict__ bad) {
  const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
  if (*bad || m >= M) return;
  const uint32_t n = mesh2tri[m + 1] - mesh2tri[m];
  if (n > 0) *packed_flag(dst[m], n) = nonfinite[m];
}

// Internal nodes of a CSR batch of trees into their packed buffers; also the
// root boxes and a per-mesh flag for boxes that need the general slab test.
static __global__ __launch_bounds__(256) void k_pack_to_buffers(
    bat::BatchTrees b, uint32_t total_tri, const uint32_t* __restrict__ inner_off,
    const uint64_t* __restrict__ dst, uint32_t* __restrict__ nonfinite,
    uint32_t* __restrict__ err) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (*b.bad || g >= total_tri) return;
  // leaves: one per triangle of the batch
  {
    const uint32_t m = bat::find_segment(b.mesh2tri, b.M, g);
    const TreeView v = bat::tree_of(b, m);
    const uint32_t k = g - b.mesh2tri[m];
    const PackedRef p = packed_ref(dst[m], v.num_leaf);
    rc::pack_leaf(p.leaf, v.bvhnodes, v.tri2vtx, v.xyz, v.num_leaf, v.num_leaf, v.num_vtx, k, err);
    if (k == 0) {
#pragma unroll
      for (int d = 0; d < 6; ++d) p.root_box[d] = v.aabb[d];
    }
  }
  // internal nodes: the first sum (N - 1) threads
  if (g < inner_off[b.M]) {
    const uint32_t m = bat::find_segment(inner_off, b.M, g);
    const TreeView v = bat::tree_of(b, m);
    const PackedRef p = packed_ref(dst[m], v.num_leaf);
    rc::pack_inner(p.inner, v.bvhnodes, v.aabb, v.num_leaf, g - inner_off[m], nonfinite + m, err);
  }
}

// One ray-cast request (the C ABI's dmsh_cast_request).
struct Request {
  uint64_t packed;
  uint32_t num_tri;
  uint32_t nonfinite;
  uint32_t img_w, img_h;
  uint32_t pix_start;
  uint32_t reserved;
  float ndc2world[16];
};
static_assert(sizeof(Request) == 96, "request layout");

// Tile and pixel offsets of the requests; rejects (counts[3], DMSH_DEVERR_INDEX)
// images that are empty or do not follow one another in pixel order.
static __global__ __launch_bounds__(1024) void k_req_offsets(uint32_t R, uint32_t total_pix,
                                                             const Request* __restrict__ req,
                                                             uint32_t* __restrict__ tile_off,
                                                             uint32_t* __restrict__ pix_off,
                                                             uint32_t* __restrict__ bad,
                                                             uint32_t* __restrict__ err) {
  bat::scan_meshes(R, pix_off, [&](uint32_t r) { return req[r].img_w * req[r].img_h; });
  bat::scan_meshes(R, tile_off, [&](uint32_t r) {
    return ceil_div_u32(req[r].img_w, 8u) * ceil_div_u32(req[r].img_h, 8u);
  });
  __syncthreads();
  for (uint32_t r = threadIdx.x; r < R; r += 1024) {
    const Request& q = req[r];
    // a running sum that wrapped past 2^32 shows up as a decrease
    const bool ok = q.img_w > 0 && q.img_h > 0 && q.pix_start == pix_off[r] &&
                    (uint64_t)q.img_w * q.img_h < (1ull << 32) && q.num_tri < rc::kMaxTri &&
                    pix_off[r + 1] > pix_off[r] && tile_off[r + 1] > tile_off[r];
    if (!ok) {
      atomicOr(bad, 1u);
      raise_error(err, DMSH_DEVERR_INDEX);
    }
  }
  if (threadIdx.x == 0 && pix_off[R] != total_pix) {
    atomicOr(bad, 1u);
    raise_error(err, DMSH_DEVERR_INDEX);
  }
}

// The images of the requests.  The general slab test is taken when the
// request or the tree says so.
struct ReqSrc {
  uint32_t R;
  const Request* req;
  const uint32_t* tile_off;  // [R + 1]
  const uint32_t* counts;
  __device__ __forceinline__ uint32_t num_tiles() const { return counts[3] ? 0u : tile_off[R]; }
  __device__ __forceinline__ bool load(uint32_t tile, uint32_t lane, rc::PixelJob& j) const {
    const uint32_t r = rc::wave_segment(tile_off, R, tile);
    const Request& q = req[r];
    const PackedRef p = packed_ref(q.packed, q.num_tri);
    j.pk = rc::Packed{p.inner, p.leaf, p.root_box, q.num_tri};
    j.T = q.ndc2world;
    j.w = q.img_w;
    j.h = q.img_h;
    const uint32_t tiles_x = ceil_div_u32(j.w, 8u), lt = tile - tile_off[r];
    j.iw = (lt % tiles_x) * 8u + (lane & 7u);
    j.ih = (lt / tiles_x) * 8u + (lane >> 3);
    j.out = q.pix_start + j.ih * j.w + j.iw;
    j.regular = q.nonfinite == 0u && (q.num_tri == 0 || *packed_flag(q.packed, q.num_tri) == 0u);
    return j.iw < j.w && j.ih < j.h;
  }
};

template <int S, int W>
__global__ __launch_bounds__(64 * W) void k_req_pix2tri(ReqSrc src, rc::CastState st,
                                                        uint32_t* __restrict__ pix2tri,
                                                        float* __restrict__ pix2t) {
  __shared__ uint64_t s_stack[W][S][64];
  rc::cast_wave<S, W>(src, st, (rc::LdsFrame*)&s_stack[threadIdx.x >> 6][0][0], pix2tri, pix2t);
}

}  // namespace srv
}  // namespace dmsh
