// batch_aa.hpp -- contours and anti-aliased silhouettes of a CSR batch of
// meshes, one launch a stage for all meshes.
//
// One mesh at a time (antialias.hpp) a step of silhouette fitting launches some
// eight kernels a mesh, most of a few microseconds, and the host cannot keep up
// with them.  Here the meshes' edges are concatenated: an edge finds its mesh in
// the offsets, the contour edges are compacted over the whole batch in edge
// order (so mesh m's are a contiguous run from mesh2cedge[m] on, in its own edge
// order), and the walks of all meshes share a launch.  The arithmetic, and the
// writes that win, are the single-mesh ones.  Eight meshes of 5,000 to 200,000
// triangles (512 x 512 images), forward and recomputing backward: 212 launches
// and 2.52 ms before, 67 and 1.57 ms now; what is left is the two casts and
// builds, and the contours and walks take 0.13 ms.
#pragma once

#include "antialias.hpp"
#include "batch.hpp"

namespace dmsh {
namespace baa {

struct ContourBatch {
  uint32_t M;
  const uint32_t* __restrict__ mesh2tri;
  const uint32_t* __restrict__ mesh2vtx;
  const uint32_t* __restrict__ tri2vtx;  // vertex ids local to each mesh
  const float* __restrict__ xyz;
  uint32_t total_edge;
  const uint32_t* __restrict__ mesh2edge;
  const uint32_t* __restrict__ edge2vtx;  // vertex and triangle ids local to each mesh
  const uint32_t* __restrict__ edge2tri;
  const float* __restrict__ w2n;  // [M][16], column-major
  float* __restrict__ n2w;        // [M][17]: inverses, and 0 for a singular one
  uint32_t* __restrict__ bad;
  uint32_t* err;
};

// Checks the offsets and inverts the transforms of the meshes that have edges
// (one workgroup).
static __global__ __launch_bounds__(1024) void k_batch_contour_init(ContourBatch b,
                                                                    uint32_t total_tri,
                                                                    uint32_t total_vtx) {
  if (threadIdx.x == 0) *b.bad = 0u;
  __syncthreads();
  bat::check_offsets(b.mesh2tri, b.M, total_tri, b.bad, b.err);
  bat::check_offsets(b.mesh2vtx, b.M, total_vtx, b.bad, b.err);
  bat::check_offsets(b.mesh2edge, b.M, b.total_edge, b.bad, b.err);
  for (uint32_t m = threadIdx.x; m < b.M; m += 1024u) {
    if (b.mesh2edge[m + 1] == b.mesh2edge[m]) continue;
    float a[16], r[16];
    for (int k = 0; k < 16; ++k) a[k] = b.w2n[(size_t)m * 16 + k];
    const bool ok = mat4_inverse(a, r);
    for (int k = 0; k < 16; ++k) b.n2w[(size_t)m * 17 + k] = r[k];
    b.n2w[(size_t)m * 17 + 16] = ok ? 1.f : 0.f;
    if (!ok) raise_error(b.err, DMSH_DEVERR_SINGULAR);
  }
}

// The contour edges as a mask a wave, counted per workgroup.
static __global__ __launch_bounds__(256) void k_batch_contour_count(
    ContourBatch b, uint64_t* __restrict__ wave_mask, uint32_t* __restrict__ block_count) {
  __shared__ uint32_t s_w[4];
  const uint32_t e = blockIdx.x * 256u + threadIdx.x;
  bool f = false;
  if (e < b.total_edge && *b.bad == 0u) {
    const uint32_t m = bat::find_segment(b.mesh2edge, b.M, e);
    const uint32_t t0 = b.mesh2tri[m], v0 = b.mesh2vtx[m], e0 = b.mesh2edge[m];
    const aa::ContourArgs a{b.tri2vtx + (size_t)t0 * 3, b.mesh2tri[m + 1] - t0,
                            b.xyz + (size_t)v0 * 3,     b.mesh2vtx[m + 1] - v0,
                            b.w2n + (size_t)m * 16,     b.n2w + (size_t)m * 17,
                            b.mesh2edge[m + 1] - e0,    b.edge2vtx + (size_t)e0 * 2,
                            b.edge2tri + (size_t)e0 * 2, b.err};
    f = aa::contour_flag(a, e - e0);
  }
  const uint64_t mask = __ballot(f);
  if ((threadIdx.x & 63u) == 0) {
    wave_mask[blockIdx.x * 4u + (threadIdx.x >> 6)] = mask;
    s_w[threadIdx.x >> 6] = (uint32_t)__popcll(mask);
  }
  __syncthreads();
  if (threadIdx.x == 0) block_count[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// Contour edges before edge e of the batch.
__device__ __forceinline__ uint32_t contour_rank(const uint64_t* __restrict__ wave_mask,
                                                 const uint32_t* __restrict__ block_offset,
                                                 uint32_t e) {
  uint32_t pos = block_offset[e >> 8];
  for (uint32_t w = (e >> 8) * 4u; w < (e >> 6); ++w) pos += (uint32_t)__popcll(wave_mask[w]);
  return pos + (uint32_t)__popcll(wave_mask[e >> 6] & ((1ull << (e & 63u)) - 1ull));
}

// Scatters the vertex pairs in edge order; the workgroups past the edges write
// where each mesh's begin.
static __global__ __launch_bounds__(256) void k_batch_contour_scatter(
    ContourBatch b, uint32_t edge_blocks, const uint64_t* __restrict__ wave_mask,
    const uint32_t* __restrict__ block_offset, uint32_t* __restrict__ mesh2cedge,
    uint32_t* __restrict__ cedge2vtx) {
  if (blockIdx.x < edge_blocks) {
    const uint32_t e = blockIdx.x * 256u + threadIdx.x;
    if (!((wave_mask[e >> 6] >> (e & 63u)) & 1ull)) return;
    const uint32_t pos = contour_rank(wave_mask, block_offset, e);
    cedge2vtx[(size_t)pos * 2] = b.edge2vtx[(size_t)e * 2];
    cedge2vtx[(size_t)pos * 2 + 1] = b.edge2vtx[(size_t)e * 2 + 1];
    return;
  }
  const uint32_t m = (blockIdx.x - edge_blocks) * 256u + threadIdx.x;
  if (m >= b.M) return;  // mesh2cedge[M] is the scan's total
  const uint32_t e = *b.bad ? 0u : b.mesh2edge[m];
  mesh2cedge[m] = e < b.total_edge ? contour_rank(wave_mask, block_offset, e) : mesh2cedge[b.M];
}

// The images and contour edges of a batch.
struct Images {
  uint32_t M;
  const uint32_t* __restrict__ mesh2vtx;
  const float* __restrict__ xyz;
  const uint32_t* __restrict__ mesh2pix;
  const uint32_t* __restrict__ mesh2width;
  uint32_t num_cedge;
  const uint32_t* __restrict__ mesh2cedge;
  const uint32_t* __restrict__ cedge2vtx;
  const float* __restrict__ w2p;  // [M][16], column-major
  const uint32_t* __restrict__ pix2tri;
  uint32_t* __restrict__ bad;
  uint32_t* err;
};

// Clears the keys (grid-strided), and checks the offsets in the last workgroup.
static __global__ __launch_bounds__(256) void k_batch_aa_init(
    Images b, uint32_t total_vtx, uint32_t total_pix, unsigned long long* __restrict__ keys,
    uint64_t num_keys) {
  if (blockIdx.x + 1u < gridDim.x) {
    for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < num_keys;
         i += (gridDim.x - 1u) * 256ull)
      keys[i] = 0ull;
    return;
  }
  if (threadIdx.x == 0) *b.bad = 0u;
  __syncthreads();
  bat::check_offsets(b.mesh2vtx, b.M, total_vtx, b.bad, b.err);
  bat::check_offsets(b.mesh2pix, b.M, total_pix, b.bad, b.err);
  bat::check_offsets(b.mesh2cedge, b.M, b.num_cedge, b.bad, b.err);
  bool ok = true;
  for (uint32_t m = threadIdx.x; m < b.M; m += 256u) {
    const uint32_t n = b.mesh2pix[m + 1] - b.mesh2pix[m], w = b.mesh2width[m];
    ok = ok && (n == 0u || (w != 0u && n % w == 0u));
  }
  if (!ok) {
    atomicOr(b.bad, 1u);
    raise_error(b.err, DMSH_DEVERR_INDEX);
  }
}

// Calls fn(the mesh's args, its contour edge, lane of the group, its first
// pixel, its first vertex) for the group's contour edge of the batch.
template <uint32_t L, class Fn>
__device__ __forceinline__ void with_cedge(const aa::EdgeSlice& es, const Images& b, Fn fn) {
  uint32_t g;
  if (!aa::group_edge<L>(es, g) || *b.bad != 0u) return;
  const uint32_t m = bat::find_segment(b.mesh2cedge, b.M, g);
  const uint32_t p0 = b.mesh2pix[m], n = b.mesh2pix[m + 1] - p0, w = b.mesh2width[m];
  if (n == 0u) return;
  const uint32_t c0 = b.mesh2cedge[m], v0 = b.mesh2vtx[m];
  const aa::EdgeArgs a{b.cedge2vtx + (size_t)c0 * 2, b.xyz + (size_t)v0 * 3,
                       b.mesh2vtx[m + 1] - v0,       b.w2p + (size_t)m * 16,
                       w,                            n / w,
                       b.pix2tri + p0,               b.err};
  fn(a, g - c0, threadIdx.x % L, p0, v0);
}

template <uint32_t L>
__global__ __launch_bounds__(64) void k_batch_aa_keys(
    aa::EdgeSlice es, Images b, unsigned long long* __restrict__ keys) {
  with_cedge<L>(es, b, [&](const aa::EdgeArgs& a, uint32_t e, uint32_t sub, uint32_t p0, uint32_t) {
    aa::keys_of_edge<L>(a, e, sub, keys + p0);
  });
}

template <uint32_t L>
__global__ __launch_bounds__(64) void k_batch_aa_write(
    aa::EdgeSlice es, Images b, const unsigned long long* __restrict__ keys,
    const float* __restrict__ vin, float* __restrict__ vout) {
  with_cedge<L>(es, b, [&](const aa::EdgeArgs& a, uint32_t e, uint32_t sub, uint32_t p0, uint32_t) {
    aa::values_of_edge<L>(a, e, sub, keys + p0, vin + p0, vout + p0);
  });
}

template <uint32_t L>
__global__ __launch_bounds__(64) void k_batch_aa_bwd(aa::EdgeSlice es, Images b,
                                                            const float* __restrict__ val,
                                                            const float* __restrict__ dldw,
                                                            float* __restrict__ dldw_vtx2xyz) {
  with_cedge<L>(es, b, [&](const aa::EdgeArgs& a, uint32_t e, uint32_t sub, uint32_t p0, uint32_t v0) {
    aa::bwd_of_edge<L>(a, e, sub, val + p0, dldw + p0, dldw_vtx2xyz + (size_t)v0 * 3);
  });
}

}  // namespace baa
}  // namespace dmsh
