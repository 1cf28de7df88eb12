"""GPU: contours and silhouettes of a batch, every stage one launch, against the
single-mesh entry points: batches smaller and larger than a workgroup of
offsets, with empty meshes, meshes without pixels and meshes without contours."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib, primitives
import del_msh_dlpack.Batched.torch as Batched
import del_msh_dlpack.DifferentiableAntialias.torch as DifferentiableAntialias
from del_msh_dlpack.Edge2Vtx import contour_for_triangle_mesh

pytestmark = pytest.mark.gpu


def _batch(num_mesh):
    """Closed meshes; of every seven, one is emptied, one loses its image and
    one is drawn together in a point, so that none of its edges is a contour."""
    b = primitives.batch_meshes(num_mesh, seed=num_mesh, tri_range=(32, 1500),
                                pix_range=(9 * 9, 90 * 90))
    ntri, nvtx, npix = (np.diff(b[k].astype(np.int64)) for k in ("mesh2tri", "mesh2vtx", "mesh2pix"))
    tri, vtx, width = [], [], b["mesh2width"].copy()
    for m in range(num_mesh):
        t = b["tri2vtx"][b["mesh2tri"][m]:b["mesh2tri"][m + 1]]
        v = b["vtx2xyz"][b["mesh2vtx"][m]:b["mesh2vtx"][m + 1]]
        if m % 7 == 1:
            t, v = t[:0], v[:0]
        elif m % 7 == 2:
            npix[m] = width[m] = 0
        elif m % 7 == 4:
            v = 0 * v
        ntri[m], nvtx[m] = len(t), len(v)
        tri.append(t)
        vtx.append(v)
    csr = lambda c: np.concatenate([[0], np.cumsum(c)]).astype(np.uint32)
    return (csr(ntri), csr(nvtx), np.concatenate(tri), np.concatenate(vtx), csr(npix), width,
            torch.from_numpy(b["ndc2world"]))


@pytest.mark.parametrize("num_mesh", [1, 8, 300])
def test_batch_equals_single_meshes(gpu, num_mesh):
    m2t, m2v, tri, vtx, m2p, width, n2w = _batch(num_mesh)
    g = lambda a: torch.from_numpy(a).to(gpu)
    t, v = g(tri), g(vtx)
    dldw = g(np.random.default_rng(1).normal(size=int(m2p[-1])).astype(np.float32))
    sb = Batched.SilhouetteBatch(m2t, m2v, t, v, m2p, width, n2w)
    hits = sb.hits(v)
    img, grad = sb.images(v, hits), sb.vertex_gradient(v, hits, dldw)
    want_img, want_grad, contours = hits["occ"].clone(), torch.zeros_like(v), 0
    for m in range(num_mesh):
        tm, vm = t[int(m2t[m]):int(m2t[m + 1])], v[int(m2v[m]):int(m2v[m + 1])]
        p = slice(int(m2p[m]), int(m2p[m + 1]))
        c = hits["cedges"][m]
        e2v, e2t = sb.edges[m]
        if e2v.shape[0] == 0:
            assert c.shape == (0, 2)
            continue
        want = contour_for_triangle_mesh(tm, vm, sb.world2ndc[m].T.contiguous().flatten(), e2v, e2t)
        assert torch.equal(c.view(torch.int32), want.view(torch.int32))
        contours += c.shape[0]
        if p.stop == p.start or c.shape[0] == 0:
            continue
        im = lambda a: a[p].view(-1, int(width[m]))
        pix, occ = im(hits["pix2tri"]), im(hits["occ"])
        want_img[p] = DifferentiableAntialias.antialias(c, vm, sb.world2pix[m], pix, occ).view(-1)
        want_grad[int(m2v[m]):int(m2v[m + 1])] = DifferentiableAntialias.bwd_antialias(
            c, vm, sb.world2pix[m], occ, im(dldw), pix)
    assert contours > 0 and not torch.equal(want_img, hits["occ"])
    assert torch.equal(img, want_img)
    # the same terms (at most 2 x 90 pairs an edge, some ten edges a vertex)
    # added in another order: each addition is off by 2^-24 of a partial sum
    bound = 1800 * 2.0 ** -24 * float(want_grad.abs().max())
    assert float((grad - want_grad).abs().max()) <= bound
    # a caller's own edges in place of the batch's
    hits["cedges"] = [c[::2].contiguous() for c in hits["cedges"]]
    half = sb.images(v, hits)
    hits["cedges"] = [c.clone() for c in sb.hits(v)["cedges"]]
    assert torch.equal(sb.images(v, hits), want_img) and not torch.equal(half, want_img)
    assert _lib.device_errors() == 0
