"""GPU: contours and silhouettes of a batch, every stage one launch, against the
single-mesh entry points: batches smaller and larger than a workgroup of
offsets, with empty meshes, meshes without pixels and meshes without contours."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib, primitives
import del_msh_dlpack.Batched.torch as Batched
import del_msh_dlpack.DifferentiableAntialias.torch as DifferentiableAntialias
from del_msh_dlpack.Edge2Vtx import contour_for_triangle_mesh, contour_for_triangle_mesh_into

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


def _single(sb, m, hits, m2v, m2p, v, dldw):
    """Image and gradient of mesh m by the single-mesh entry points."""
    p = slice(int(m2p[m]), int(m2p[m + 1]))
    vm, c = v[int(m2v[m]):int(m2v[m + 1])], hits["cedges"][m]
    im = lambda a: a[p].view(*sb.shapes[m])
    pix, occ = im(hits["pix2tri"]), im(hits["occ"])
    return (DifferentiableAntialias.antialias(c, vm, sb.world2pix[m], pix, occ).view(-1),
            DifferentiableAntialias.bwd_antialias(c, vm, sb.world2pix[m], occ, im(dldw), pix))


REPLACED = [(what, how) for what in ("world2ndc", "world2pix", "edges", "shapes")
            for how in ("entry", "list")]
REPLACED += [("world2ndc", "in place"), ("world2ndc", "data"), ("world2pix", "in place"),
             ("world2pix", "data"), ("edges", "data")]


@pytest.mark.parametrize("what,how", REPLACED)
def test_replaced_entries_are_used(gpu, what, how):
    """Another camera, other edges or another image shape in place of a mesh's
    own, by whichever way the caller puts it there."""
    m2t, m2v, tri, vtx, m2p, width, n2w = _batch(5)
    g = lambda a: torch.from_numpy(a).to(gpu)
    t, v = g(tri), g(vtx)
    dldw = g(np.random.default_rng(1).normal(size=int(m2p[-1])).astype(np.float32))
    sb = Batched.SilhouetteBatch(m2t, m2v, t, v, m2p, width, n2w)
    before = sb.hits(v)
    img_before = sb.images(v, before)
    m = 3
    if what == "edges":
        new = tuple(e[::3].contiguous() for e in sb.edges[m])
    elif what == "shapes":
        new = (1, sb.shapes[m][0] * sb.shapes[m][1])
    else:  # the mesh turned about x and moved aside
        turn = torch.tensor([[1, 0, 0, 0.1], [0, 0.8, -0.6, 0], [0, 0.6, 0.8, 0], [0, 0, 0, 1.0]])
        new = (getattr(sb, what)[m].cpu() @ turn).to(gpu)
    entries = getattr(sb, what)
    if how == "entry":
        entries[m] = new
    elif how == "list":
        setattr(sb, what, [new if k == m else e for k, e in enumerate(entries)])
    elif how == "in place":
        entries[m].copy_(new)
    else:
        for old, data in zip(entries[m], new) if what == "edges" else [(entries[m], new)]:
            old.data = data
    hits = sb.hits(v)
    for k in range(5):
        if sb.edges[k][0].shape[0] == 0:
            continue
        want = contour_for_triangle_mesh(
            t[int(m2t[k]):int(m2t[k + 1])], v[int(m2v[k]):int(m2v[k + 1])],
            sb.world2ndc[k].T.contiguous().flatten(), *sb.edges[k])
        assert torch.equal(hits["cedges"][k].view(torch.int32), want.view(torch.int32))
    same = torch.equal(hits["cedges"][m].view(torch.int32), before["cedges"][m].view(torch.int32))
    assert same == (what in ("world2pix", "shapes"))
    img, grad = sb.images(v, hits), sb.vertex_gradient(v, hits, dldw)
    want_img, want_grad = _single(sb, m, hits, m2v, m2p, v, dldw)
    p, q = slice(int(m2p[m]), int(m2p[m + 1])), slice(int(m2v[m]), int(m2v[m + 1]))
    assert torch.equal(img[p], want_img) and not torch.equal(img[p], img_before[p])
    assert torch.equal(img[:p.start], img_before[:p.start])
    # the bound of test_batch_equals_single_meshes
    assert float((grad[q] - want_grad).abs().max()) <= 1800 * 2.0 ** -24 * float(want_grad.abs().max())
    assert _lib.device_errors() == 0


def test_broken_rows_of_an_image_without_contours(gpu):
    """An image whose pixels are not whole rows stops only a call that has to
    walk its contour edges."""
    m2t, m2v, tri, vtx, m2p, width, n2w = _batch(4)
    g = lambda a: torch.from_numpy(a).to(gpu)
    t, v = g(tri), g(vtx)
    dldw = g(np.random.default_rng(1).normal(size=int(m2p[-1])).astype(np.float32))
    whole = Batched.SilhouetteBatch(m2t, m2v, t, v, m2p, width, n2w)
    hits = whole.hits(v)
    want = whole.images(v, hits), whole.vertex_gradient(v, hits, dldw)
    for m, ok in ((1, True), (3, False)):  # the emptied mesh, and one with contours
        broken = width.copy()
        broken[m] += 1
        assert int(m2p[m + 1] - m2p[m]) % int(broken[m]) != 0
        sb = Batched.SilhouetteBatch(m2t, m2v, t, v, m2p, broken, n2w)
        if ok:
            assert torch.equal(sb.images(v, hits), want[0])
            # the bound of test_batch_equals_single_meshes
            bound = 1800 * 2.0 ** -24 * float(want[1].abs().max())
            assert float((sb.vertex_gradient(v, hits, dldw) - want[1]).abs().max()) <= bound
        else:
            for call in (lambda: sb.images(v, hits), lambda: sb.vertex_gradient(v, hits, dldw)):
                with pytest.raises(RuntimeError):
                    call()
    assert _lib.device_errors() == 0


def test_contours_into_a_callers_buffers(gpu):
    """contour_for_triangle_mesh_into: several meshes' contours back to back
    without a read in between, in a workspace for the largest."""
    m2t, m2v, tri, vtx, m2p, width, n2w = _batch(6)
    g = lambda a: torch.from_numpy(a).to(gpu)
    t, v = g(tri), g(vtx)
    sb = Batched.SilhouetteBatch(m2t, m2v, t, v, m2p, width, n2w)
    live = [m for m in range(6) if sb.edges[m][0].shape[0]]
    size = [sb.edges[m][0].shape[0] for m in live]
    ws = _lib.workspace(_lib.lib().dmsh_contour_workspace_bytes(max(size)), gpu)
    count = torch.zeros(len(live), dtype=torch.uint32, device=gpu)
    out = [torch.empty((n, 2), dtype=torch.uint32, device=gpu) for n in size]
    args = [(t[int(m2t[m]):int(m2t[m + 1])], v[int(m2v[m]):int(m2v[m + 1])],
             sb.world2ndc[m].T.contiguous().flatten(), *sb.edges[m]) for m in live]
    for k, a in enumerate(args):
        contour_for_triangle_mesh_into(*a, out[k], count[k:k + 1], ws)
    for n, c, a in zip(count.cpu().numpy().tolist(), out, args):
        want = contour_for_triangle_mesh(*a)
        assert torch.equal(c[:n].view(torch.int32), want.view(torch.int32))
    assert _lib.device_errors() == 0
