// dmsh_aa.hip -- C ABI: contour edges and the anti-aliased silhouette.
#include <algorithm>
#include <type_traits>

#include "antialias.hpp"
#include "batch_aa.hpp"

using namespace dmsh;

namespace {

struct ContourLayout {
  float* n2w;  // 16 + ok flag
  uint32_t* flags;
  uint32_t* block_count;
};

// Launches a kernel over num_cedge contour edges in blocks of 64 threads, `lanes`
// an edge.
template <typename... KArgs, typename... Args>
int launch_edges(const char* label, void (*kernel)(aa::EdgeSlice, KArgs...), uint32_t lanes,
                 uint32_t num_cedge, hipStream_t s, const Args&... args) {
  int st = DMSH_OK;
  for (aa::EdgeSlice es{0u, 0u}; st == DMSH_OK && es.first < num_cedge; es.first += es.count) {
    es.count = std::min(num_cedge - es.first, aa::kEdgeSlice);
    launch(label, kernel, dim3(ceil_div(es.count, 64u / lanes)), dim3(64), 0, s, es, args...);
    st = launch_status();
  }
  return st;
}

// Calls fn(integral_constant of the lanes an edge).
template <class Fn>
int with_lanes(uint32_t num_cedge, bool backward, Fn fn) {
  switch (aa::edge_lanes(num_cedge, backward)) {
    case 16: return fn(std::integral_constant<uint32_t, 16>());
    case 8: return fn(std::integral_constant<uint32_t, 8>());
    default: return fn(std::integral_constant<uint32_t, 4>());
  }
}

inline uint32_t contour_blocks(uint32_t num_edge) { return ceil_div(num_edge, 256); }

inline bool carve_contour(Arena& a, uint32_t num_edge, ContourLayout& L) {
  L.n2w = a.take<float>(17);
  L.flags = a.take<uint32_t>(num_edge ? num_edge : 1);
  L.block_count = a.take<uint32_t>(num_edge ? contour_blocks(num_edge) : 1);
  return a.ok();
}

struct BatchContourLayout {
  float* n2w;
  uint64_t* wave_mask;
  uint32_t* block_count;
  uint32_t* bad;
};

inline bool carve_batch_contour(Arena& a, uint32_t num_mesh, uint32_t total_edge,
                                BatchContourLayout& L) {
  const uint32_t nb = contour_blocks(total_edge);
  L.n2w = a.take<float>((size_t)num_mesh * 17);
  L.wave_mask = a.take<uint64_t>((size_t)nb * 4 + 1);
  L.block_count = a.take<uint32_t>((size_t)nb + 1);
  L.bad = a.take<uint32_t>(1);
  return a.ok();
}

struct BatchAaLayout {
  unsigned long long* keys;
  uint32_t* bad;
};

inline bool carve_batch_aa(Arena& a, uint32_t total_pix, BatchAaLayout& L) {
  L.keys = a.take<unsigned long long>((size_t)total_pix + 1);
  L.bad = a.take<uint32_t>(1);
  return a.ok();
}

}  // namespace

extern "C" {

size_t dmsh_contour_workspace_bytes(uint32_t num_edge) {
  Arena a{nullptr, ~(size_t)0, 0};
  ContourLayout L;
  carve_contour(a, num_edge, L);
  return a.off + 256;
}

int dmsh_contour_for_triangle_mesh(void* stream, uint32_t num_tri, const uint32_t* tri2vtx,
                                   uint32_t num_vtx, const float* vtx2xyz,
                                   const float* transform_world2ndc, uint32_t num_edge,
                                   const uint32_t* edge2vtx, const uint32_t* edge2tri,
                                   uint32_t* cedge2vtx, uint32_t* num_cedge, void* ws,
                                   size_t ws_bytes) {
  if (!num_cedge || !transform_world2ndc) return DMSH_ERR_INVALID;
  if (num_edge > 0 && (!tri2vtx || !vtx2xyz || !edge2vtx || !edge2tri || !cedge2vtx))
    return DMSH_ERR_INVALID;
  if (!ws || ws_bytes < dmsh_contour_workspace_bytes(num_edge)) return DMSH_ERR_WORKSPACE;
  uint32_t* err = device_error_word();
  if (!err) return DMSH_ERR_HIP;
  hipStream_t s = as_stream(stream);
  Arena a{static_cast<char*>(ws), ws_bytes, 0};
  ContourLayout L;
  if (!carve_contour(a, num_edge, L)) return DMSH_ERR_WORKSPACE;
  launch("k_mat4_inverse", k_mat4_inverse, dim3(1), dim3(1), 0, s, transform_world2ndc, L.n2w, err);
  int st = launch_status();
  if (st != DMSH_OK) return st;
  const uint32_t nb = num_edge ? contour_blocks(num_edge) : 0;
  if (nb) {
    aa::ContourArgs ca{tri2vtx, num_tri, vtx2xyz, num_vtx, transform_world2ndc, L.n2w,
                       num_edge, edge2vtx, edge2tri, err};
    launch("k_contour_count", aa::k_contour_count, dim3(nb), dim3(256), 0, s, ca, L.flags,
                       L.block_count);
    if ((st = launch_status()) != DMSH_OK) return st;
  }
  // also writes the total when there is no edge (0)
  launch("k_scan_counts", aa::k_scan_counts, dim3(1), dim3(1024), 0, s, L.block_count, nb, num_cedge);
  if ((st = launch_status()) != DMSH_OK) return st;
  if (nb) {
    launch("k_contour_scatter", aa::k_contour_scatter, dim3(nb), dim3(256), 0, s, edge2vtx, num_edge,
                       L.flags, L.block_count, cedge2vtx);
    st = launch_status();
  }
  return st;
}

size_t dmsh_antialias_workspace_bytes(uint32_t img_w, uint32_t img_h) {
  return (size_t)img_w * img_h * sizeof(unsigned long long) + 256;
}

int dmsh_antialias_fwd(void* stream, uint32_t num_cedge, const uint32_t* cedge2vtx,
                       uint32_t num_vtx, const float* vtx2xyz, const float* transform_world2pix,
                       uint32_t img_w, uint32_t img_h, const uint32_t* pix2tri,
                       const float* pix2vin, float* pix2vout, void* ws, size_t ws_bytes) {
  const uint64_t num_pix = (uint64_t)img_w * img_h;
  if (num_pix == 0 || num_cedge == 0) return DMSH_OK;
  if (num_pix >= (1ull << 32) || num_cedge == DMSH_U32MAX) return DMSH_ERR_INVALID;
  if (!cedge2vtx || !vtx2xyz || !transform_world2pix || !pix2tri || !pix2vin || !pix2vout)
    return DMSH_ERR_INVALID;
  if (!ws || ws_bytes < dmsh_antialias_workspace_bytes(img_w, img_h)) return DMSH_ERR_WORKSPACE;
  uint32_t* err = device_error_word();
  if (!err) return DMSH_ERR_HIP;
  hipStream_t s = as_stream(stream);
  auto* keys = static_cast<unsigned long long*>(ws);
  launch("k_zero_u64", aa::k_zero_u64, dim3(std::min<uint32_t>(ceil_div(num_pix, 256), 4096)),
                     dim3(256), 0, s, keys, num_pix);
  int st = launch_status();
  if (st != DMSH_OK) return st;
  const aa::EdgeArgs ea{cedge2vtx, vtx2xyz, num_vtx, transform_world2pix,
                        img_w, img_h, pix2tri, err};
  return with_lanes(num_cedge, false, [&](auto lanes) {
    constexpr uint32_t L = decltype(lanes)::value;
    const int rc = launch_edges("k_aa_keys", aa::k_aa_keys<L>, L, num_cedge, s, ea, keys);
    if (rc != DMSH_OK) return rc;
    return launch_edges("k_aa_write", aa::k_aa_write<L>, L, num_cedge, s, ea, keys, pix2vin,
                        pix2vout);
  });
}

int dmsh_antialias_bwd(void* stream, uint32_t num_cedge, const uint32_t* cedge2vtx,
                       uint32_t num_vtx, const float* vtx2xyz, float* dldw_vtx2xyz,
                       const float* transform_world2pix, uint32_t img_w, uint32_t img_h,
                       const float* pix2val, const float* dldw_pix2val, const uint32_t* pix2tri) {
  const uint64_t num_pix = (uint64_t)img_w * img_h;
  if (num_pix == 0 || num_cedge == 0) return DMSH_OK;
  if (num_pix >= (1ull << 32) || num_cedge == DMSH_U32MAX) return DMSH_ERR_INVALID;
  if (!cedge2vtx || !vtx2xyz || !dldw_vtx2xyz || !transform_world2pix || !pix2val ||
      !dldw_pix2val || !pix2tri)
    return DMSH_ERR_INVALID;
  uint32_t* err = device_error_word();
  if (!err) return DMSH_ERR_HIP;
  const aa::EdgeArgs ea{cedge2vtx, vtx2xyz, num_vtx, transform_world2pix,
                        img_w, img_h, pix2tri, err};
  return with_lanes(num_cedge, true, [&](auto lanes) {
    constexpr uint32_t L = decltype(lanes)::value;
    return launch_edges("k_aa_bwd", aa::k_aa_bwd<L>, L, num_cedge, as_stream(stream), ea, pix2val,
                        dldw_pix2val, dldw_vtx2xyz);
  });
}

size_t dmsh_batch_contour_workspace_bytes(uint32_t num_mesh, uint32_t total_edge) {
  Arena a{nullptr, ~(size_t)0, 0};
  BatchContourLayout L;
  carve_batch_contour(a, num_mesh, total_edge, L);
  return a.off + 256;
}

int dmsh_batch_contour(void* stream, uint32_t num_mesh, uint32_t total_tri, uint32_t total_vtx,
                       uint32_t total_edge, const uint32_t* mesh2tri, const uint32_t* mesh2vtx,
                       const uint32_t* tri2vtx, const float* vtx2xyz,
                       const float* transforms_world2ndc, const uint32_t* mesh2edge,
                       const uint32_t* edge2vtx, const uint32_t* edge2tri, uint32_t* mesh2cedge,
                       uint32_t* cedge2vtx, void* ws, size_t ws_bytes) {
  if (num_mesh == 0 || !mesh2tri || !mesh2vtx || !mesh2edge || !transforms_world2ndc || !mesh2cedge)
    return DMSH_ERR_INVALID;
  if (total_edge > 0 && (!tri2vtx || !vtx2xyz || !edge2vtx || !edge2tri || !cedge2vtx))
    return DMSH_ERR_INVALID;
  if (!ws || ws_bytes < dmsh_batch_contour_workspace_bytes(num_mesh, total_edge))
    return DMSH_ERR_WORKSPACE;
  Arena ar{static_cast<char*>(ws), ws_bytes, 0};
  BatchContourLayout L;
  if (!carve_batch_contour(ar, num_mesh, total_edge, L)) return DMSH_ERR_WORKSPACE;
  uint32_t* err = device_error_word();
  if (!err) return DMSH_ERR_HIP;
  hipStream_t s = as_stream(stream);
  const uint32_t nb = contour_blocks(total_edge);
  const baa::ContourBatch b{num_mesh,  mesh2tri, mesh2vtx, tri2vtx,
                            vtx2xyz,   total_edge, mesh2edge, edge2vtx,
                            edge2tri,  transforms_world2ndc, L.n2w, L.bad, err};
  launch("k_batch_contour_init", baa::k_batch_contour_init, dim3(1), dim3(1024), 0, s, b,
         total_tri, total_vtx);
  int st = launch_status();
  if (st != DMSH_OK) return st;
  if (nb) {
    launch("k_batch_contour_count", baa::k_batch_contour_count, dim3(nb), dim3(256), 0, s, b,
           L.wave_mask, L.block_count);
    if ((st = launch_status()) != DMSH_OK) return st;
  }
  // also writes the total when there is no edge (0)
  launch("k_scan_counts", aa::k_scan_counts, dim3(1), dim3(1024), 0, s, L.block_count, nb,
         mesh2cedge + num_mesh);
  if ((st = launch_status()) != DMSH_OK) return st;
  launch("k_batch_contour_scatter", baa::k_batch_contour_scatter,
         dim3(nb + ceil_div(num_mesh, 256)), dim3(256), 0, s, b, nb, L.wave_mask, L.block_count,
         mesh2cedge, cedge2vtx);
  return launch_status();
}

size_t dmsh_batch_antialias_workspace_bytes(uint32_t total_pix) {
  Arena a{nullptr, ~(size_t)0, 0};
  BatchAaLayout L;
  carve_batch_aa(a, total_pix, L);
  return a.off + 256;
}

int dmsh_batch_antialias_fwd(void* stream, uint32_t num_mesh, uint32_t total_vtx,
                             uint32_t total_pix, uint32_t num_cedge, const uint32_t* mesh2vtx,
                             const float* vtx2xyz, const uint32_t* mesh2pix,
                             const uint32_t* mesh2width, const uint32_t* mesh2cedge,
                             const uint32_t* cedge2vtx, const float* transforms_world2pix,
                             const uint32_t* pix2tri, const float* pix2vin, float* pix2vout,
                             void* ws, size_t ws_bytes) {
  if (total_pix == 0 || num_cedge == 0) return DMSH_OK;
  if (num_mesh == 0 || num_cedge == DMSH_U32MAX) return DMSH_ERR_INVALID;
  if (!mesh2vtx || !vtx2xyz || !mesh2pix || !mesh2width || !mesh2cedge || !cedge2vtx ||
      !transforms_world2pix || !pix2tri || !pix2vin || !pix2vout)
    return DMSH_ERR_INVALID;
  if (!ws || ws_bytes < dmsh_batch_antialias_workspace_bytes(total_pix)) return DMSH_ERR_WORKSPACE;
  Arena ar{static_cast<char*>(ws), ws_bytes, 0};
  BatchAaLayout L;
  if (!carve_batch_aa(ar, total_pix, L)) return DMSH_ERR_WORKSPACE;
  uint32_t* err = device_error_word();
  if (!err) return DMSH_ERR_HIP;
  hipStream_t s = as_stream(stream);
  const baa::Images b{num_mesh,   mesh2vtx,  vtx2xyz,              mesh2pix, mesh2width, num_cedge,
                      mesh2cedge, cedge2vtx, transforms_world2pix, pix2tri,  L.bad,      err};
  launch("k_batch_aa_init", baa::k_batch_aa_init,
         dim3(std::min<uint32_t>(ceil_div(total_pix, 256), 4096) + 1), dim3(256), 0, s, b,
         total_vtx, total_pix, L.keys, (uint64_t)total_pix);
  int st = launch_status();
  if (st != DMSH_OK) return st;
  return with_lanes(num_cedge, false, [&](auto lanes) {
    constexpr uint32_t N = decltype(lanes)::value;
    const int rc =
        launch_edges("k_batch_aa_keys", baa::k_batch_aa_keys<N>, N, num_cedge, s, b, L.keys);
    if (rc != DMSH_OK) return rc;
    return launch_edges("k_batch_aa_write", baa::k_batch_aa_write<N>, N, num_cedge, s, b, L.keys,
                        pix2vin, pix2vout);
  });
}

int dmsh_batch_antialias_bwd(void* stream, uint32_t num_mesh, uint32_t total_vtx,
                             uint32_t total_pix, uint32_t num_cedge, const uint32_t* mesh2vtx,
                             const float* vtx2xyz, float* dldw_vtx2xyz, const uint32_t* mesh2pix,
                             const uint32_t* mesh2width, const uint32_t* mesh2cedge,
                             const uint32_t* cedge2vtx, const float* transforms_world2pix,
                             const float* pix2val, const float* dldw_pix2val,
                             const uint32_t* pix2tri, void* ws, size_t ws_bytes) {
  if (total_pix == 0 || num_cedge == 0) return DMSH_OK;
  if (num_mesh == 0 || num_cedge == DMSH_U32MAX) return DMSH_ERR_INVALID;
  if (!mesh2vtx || !vtx2xyz || !dldw_vtx2xyz || !mesh2pix || !mesh2width || !mesh2cedge ||
      !cedge2vtx || !transforms_world2pix || !pix2val || !dldw_pix2val || !pix2tri)
    return DMSH_ERR_INVALID;
  if (!ws || ws_bytes < dmsh_batch_antialias_workspace_bytes(0)) return DMSH_ERR_WORKSPACE;
  Arena ar{static_cast<char*>(ws), ws_bytes, 0};
  BatchAaLayout L;
  if (!carve_batch_aa(ar, 0, L)) return DMSH_ERR_WORKSPACE;
  uint32_t* err = device_error_word();
  if (!err) return DMSH_ERR_HIP;
  hipStream_t s = as_stream(stream);
  const baa::Images b{num_mesh,   mesh2vtx,  vtx2xyz,              mesh2pix, mesh2width, num_cedge,
                      mesh2cedge, cedge2vtx, transforms_world2pix, pix2tri,  L.bad,      err};
  launch("k_batch_aa_init", baa::k_batch_aa_init, dim3(1), dim3(256), 0, s, b, total_vtx,
         total_pix, L.keys, (uint64_t)0);
  int st = launch_status();
  if (st != DMSH_OK) return st;
  return with_lanes(num_cedge, true, [&](auto lanes) {
    constexpr uint32_t N = decltype(lanes)::value;
    return launch_edges("k_batch_aa_bwd", baa::k_batch_aa_bwd<N>, N, num_cedge, s, b, pix2val,
                        dldw_pix2val, dldw_vtx2xyz);
  });
}

}  // extern "C"
