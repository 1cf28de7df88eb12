"""GPU: the ordered edge gradient at image sizes around whole workgroups of
pixel pairs and more of them than one scan round holds, against the oracle."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib, primitives
import del_msh_dlpack.Pix2Tri.torch as Pix2Tri
import del_msh_dlpack.RasterizedEdgeGradient.torch as RasterizedEdgeGradient
import del_msh_dlpack.TriMesh3.torch as TriMesh3

pytestmark = pytest.mark.gpu


# 1100 x 1000: 8590 workgroups of 256 pairs, a scan round holds 8192
@pytest.mark.parametrize("w, h", [(1, 40), (40, 1), (2, 2), (16, 8), (16, 9), (65, 33), (1100, 1000)])
@pytest.mark.parametrize("channels", [1, 3])
def test_ordered_gradient_equals_oracle(gpu, oracle, w, h, channels):
    tri, vtx = primitives.torus_zup(1.0, 0.35, 20, 10)
    tri = tri.astype(np.uint32)
    vtx = (vtx.astype(np.float64) @ np.array([[1, 0, 0], [0, 0.7, -0.7], [0, 0.7, 0.7]]).T).astype(np.float32)
    w2n = np.diag([0.7, 0.7, 0.35, 1.0])
    n2p = np.array([[0.5 * w, 0, 0, 0.5 * w], [0, -0.5 * h, 0, 0.5 * h], [0, 0, 0.5, 0.5], [0, 0, 0, 1]])
    w2p = (n2p @ w2n).astype(np.float32)
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    t, v = g(tri), g(vtx)
    nodes, boxes = TriMesh3.make_bvhnodes_bvhnode2aabb(t, v)
    pix = Pix2Tri.by_raycasting(t, v, nodes, boxes, g(np.linalg.inv(w2n).astype(np.float32)), (w, h))
    rng = np.random.default_rng(w + h)
    val = rng.random((h, w, channels), dtype=np.float32)
    dldw = rng.normal(size=(h, w, channels)).astype(np.float32)
    got = RasterizedEdgeGradient.bwd(t, v, g(w2p), pix, g(val), g(dldw)).cpu().numpy()
    want = oracle.edge_gradient_bwd(tri, vtx, oracle.colmajor(w2p), pix.cpu().numpy(), val, dldw)
    assert min(w, h) <= 2 or np.abs(want).max() > 0
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert _lib.device_errors() == 0
