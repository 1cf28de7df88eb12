"""GPU: contour edges walked by groups of lanes, over lengths around whole
rounds of a group and walks that start, end or run outside the image, against
the oracle's serial walk."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib
import del_msh_dlpack.Batched.torch as Batched
import del_msh_dlpack.DifferentiableAntialias.torch as DifferentiableAntialias

pytestmark = pytest.mark.gpu

W, H = 150, 90


def _edges(rng):
    """Edges in pixel coordinates: (2 n, 3) vertices, (n, 2) edges."""
    ends = []
    for length in (0.0, 0.3, 1.0, 14.5, 15.0, 15.5, 16.0, 16.5, 31.0, 32.0, 33.0, 48.2, 120.0):
        for angle in np.concatenate([np.arange(8) * np.pi / 4, rng.uniform(0, 6.3, 4)]):
            p = rng.uniform((-20, -20), (W + 20, H + 20))
            ends += [p, p + length * np.array([np.cos(angle), np.sin(angle)])]
    ends += [np.array([-500.0, 40.2]), np.array([700.0, 41.7]), np.array([60.5, 20.0]),
             np.array([np.inf, 3.0])]
    vtx = np.zeros((len(ends), 3), np.float32)
    vtx[:, :2] = np.array(ends)
    return vtx, np.arange(len(ends), dtype=np.uint32).reshape(-1, 2)


# edges that are skipped, after the others, so that sixteen, eight and four lanes
# walk an edge
@pytest.mark.parametrize("more", [0, (1 << 14) + 1, (1 << 16) + 1, (1 << 18) + 1])
@pytest.mark.parametrize("seed", [0, 1])
@pytest.mark.parametrize("cover", [0.5, 0.95])
def test_walks_equal_the_serial_walk(gpu, oracle, seed, cover, more):
    rng = np.random.default_rng(seed)
    vtx, edge = _edges(rng)
    assert not np.isfinite(vtx[-1]).all()
    edge = np.concatenate([edge, np.full((more, 2), len(vtx) - 1, np.uint32)])
    pix = np.where(rng.random((H, W)) < cover, 3, 0xFFFFFFFF).astype(np.uint32)
    val = rng.random((H, W), dtype=np.float32)
    dldw = rng.normal(size=(H, W)).astype(np.float32)
    eye = np.eye(4, dtype=np.float32)
    g = lambda a: torch.from_numpy(a).to(gpu)
    got = DifferentiableAntialias.antialias(g(edge), g(vtx), g(eye), g(pix), g(val))
    want = oracle.antialias(edge, vtx, eye.reshape(-1), pix, val)
    assert not np.array_equal(want, val)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
    got = DifferentiableAntialias.bwd_antialias(g(edge), g(vtx), g(eye), g(val), g(dldw), g(pix))
    want = oracle.bwd_antialias(edge, vtx, eye.reshape(-1), val, dldw, pix)
    got = got.cpu().numpy()
    # up to 4 x 120 terms an edge in another order, the finite ones: each
    # addition is off by 2^-24 of a partial sum, and those stay within a few
    # times the largest gradient
    assert np.abs(got - want).max() <= 480 * 2.0 ** -24 * 4 * np.abs(want).max()
    assert _lib.device_errors() == 0


def test_edges_past_one_launch(gpu):
    """More edges than a launch has groups of lanes: the first and the last ones
    are real, those between have a vertex that is not finite and are skipped."""
    rng = np.random.default_rng(2)
    vtx, edge = _edges(rng)
    skipped = len(vtx) - 1
    assert not np.isfinite(vtx[skipped]).all()
    g = lambda a: torch.from_numpy(a).to(gpu)
    many = torch.full((2 ** 28 + 3, 2), skipped, dtype=torch.int32, device=gpu)
    half = len(edge) // 2
    many[:half] = g(edge[:half].view(np.int32))
    many[half - len(edge):] = g(edge[half:].view(np.int32))
    many = many.view(torch.uint32)
    pix = g(np.where(rng.random((H, W)) < 0.8, 3, 0xFFFFFFFF).astype(np.uint32))
    val = g(rng.random((H, W), dtype=np.float32))
    dldw = g(rng.normal(size=(H, W)).astype(np.float32))
    eye, v = torch.eye(4, device=gpu), g(vtx)
    want = DifferentiableAntialias.antialias(g(edge), v, eye, pix, val)
    assert not torch.equal(want, val)
    assert torch.equal(DifferentiableAntialias.antialias(many, v, eye, pix, val), want)
    want_grad = DifferentiableAntialias.bwd_antialias(g(edge), v, eye, val, dldw, pix)
    grad = DifferentiableAntialias.bwd_antialias(many, v, eye, val, dldw, pix)
    # the bound of the test above
    bound = 480 * 2.0 ** -24 * 4 * float(want_grad.abs().max())
    assert float((grad - want_grad).abs().max()) <= bound
    # and as a batch of one mesh with an image of its own
    tri = torch.zeros((1, 3), dtype=torch.uint32, device=gpu)
    sb = Batched.SilhouetteBatch([0, 1], [0, len(vtx)], tri, v, [0, W * H], [W],
                                 torch.eye(4)[None])
    sb.world2pix[0] = eye
    hits = {"pix2tri": pix.view(-1), "occ": val.view(-1), "cedges": [many]}
    assert torch.equal(sb.images(v, hits), want.view(-1))
    grad = sb.vertex_gradient(v, hits, dldw.view(-1))
    assert float((grad - want_grad).abs().max()) <= bound
    assert _lib.device_errors() == 0
