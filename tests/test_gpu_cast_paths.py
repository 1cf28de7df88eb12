"""GPU: the ray-cast where its stack leaves LDS and where its regular slab test
meets parallel axes on a box's plane, against the oracle bit for bit."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib, primitives
import del_msh_dlpack.Batched.torch as Batched
import del_msh_dlpack.Pix2Tri.torch as Pix2Tri

pytestmark = pytest.mark.gpu


def _cast_equals_oracle(gpu, oracle, tri, vtx, n2w, w, h):
    bn, aabb = oracle.build_trimesh3(tri, vtx)
    dev = [torch.from_numpy(a).to(gpu) for a in (tri, vtx, bn, aabb, n2w)]
    pix, t = Pix2Tri.by_raycasting_with_coeff(*dev, (w, h))
    want, want_t, _ = oracle.pix2tri(tri, vtx, bn, aabb, n2w.T.reshape(-1), w, h, num_threads=4)
    assert np.array_equal(pix.cpu().numpy(), want)
    assert np.array_equal(t.cpu().numpy().view(np.uint32), want_t.view(np.uint32))
    assert _lib.device_errors() == 0
    return want


def _sheets(count):
    """Sheets in one Morton cell, listed far to near, that put a frame on the
    stack for every sheet."""
    tri, vtx = [], []
    for k in range(count):
        z = -0.001 + k * (0.0016 / count)
        tri.append([len(vtx), len(vtx) + 1, len(vtx) + 2])
        vtx += [[-0.5, -0.5, z], [0.6, -0.45, z], [-0.45, 0.6, z]]
    for s in (-1.0, 1.0):
        tri.append([len(vtx), len(vtx) + 1, len(vtx) + 2])
        vtx += [[s * 4, s * 4, 0], [s * 4 + 0.01, s * 4, 0], [s * 4, s * 4 + 0.01, 0]]
    return np.array(tri, np.uint32), np.array(vtx, np.float32)


# 12 frames in LDS, 60 more in the spill area by sixes, then a lone lane's stack
@pytest.mark.parametrize("sheets", [11, 12, 13, 14, 18, 19, 20, 25, 60, 71, 72, 73, 74, 77, 79, 200])
@pytest.mark.parametrize("size", [(8, 8), (33, 17)])
def test_stack_beyond_lds_and_spill(gpu, oracle, sheets, size):
    want = _cast_equals_oracle(gpu, oracle, *_sheets(sheets), np.eye(4, dtype=np.float32), *size)
    assert (want == sheets - 1).any()


@pytest.mark.parametrize("waves", [1, 2, 4])
@pytest.mark.parametrize("stack", [12, 16, 32])
def test_stacks_of_wide_workgroups(gpu, oracle, waves, stack):
    """Waves that share a workgroup keep their frames apart, in LDS, in the spill
    area and as lone lanes, in every cast: images whose number of tiles is no
    multiple of the waves, rays that need 10 to 200 frames in all waves at once."""
    meshes = [_sheets(k) for k in (10, 20, 70, 90, 200)]
    sizes = [(41, 29), (8, 8), (57, 57), (23, 100), (64, 9)]
    eye = np.eye(4, dtype=np.float32)
    csr = lambda n: np.concatenate([[0], np.cumsum(n)]).astype(np.uint32)
    m2t, m2v = csr([len(t) for t, _ in meshes]), csr([len(v) for _, v in meshes])
    m2p = csr([w * h for w, h in sizes])
    tri, vtx = (torch.from_numpy(np.concatenate(a)).to(gpu) for a in zip(*meshes))
    L = _lib.lib()
    keys = ((L.dmsh_set_tuning, L.dmsh_get_tuning, b"pix2tri.waves", waves),
            (L.dmsh_set_tuning, L.dmsh_get_tuning, b"pix2tri.stack", stack),
            (L.dmsh_batch_set_tuning, L.dmsh_batch_get_tuning, b"batch.cast_waves", waves),
            (L.dmsh_batch_set_tuning, L.dmsh_batch_get_tuning, b"batch.stack", stack))
    old = [get(key) for _, get, key, _ in keys]
    try:
        for put, _, key, value in keys:
            assert put(key, value) == 0
        want = [_cast_equals_oracle(gpu, oracle, *mesh, eye, *size)
                for mesh, size in zip(meshes, sizes)]
        for packed in (False, True):
            p = Batched.Pipeline(m2t, m2v, tri, vtx, m2p, [w for w, _ in sizes],
                                 torch.eye(4).repeat(len(sizes), 1, 1), packed=packed)
            p.run()
            for m, image in enumerate(want):
                assert np.array_equal(p.mesh_image(m)[0].cpu().numpy(), image)
    finally:
        for (put, _, key, _), value in zip(keys, old):
            assert put(key, value) == 0
    assert _lib.device_errors() == 0


@pytest.mark.parametrize("flip", [(1, 1, 1), (-1, 1, 1), (1, 1, -1)])
@pytest.mark.parametrize("seed", [0, 1])
def test_rays_in_box_planes(gpu, oracle, flip, seed):
    """Axis-aligned quads whose edges lie at the pixel centres of an
    orthographic camera: every ray has two parallel axes and runs in the planes
    of many boxes (lo == o, hi == o, flat boxes)."""
    rng = np.random.default_rng(seed)
    w = 32
    at = lambda i: 2.0 * (i + 0.5) / w - 1.0
    tri, vtx = [], []
    for _ in range(300):
        x0, y0 = rng.integers(0, w - 1, 2)
        x1, y1 = x0 + rng.integers(1, 6), y0 + rng.integers(1, 6)
        z = rng.integers(-8, 8) / 8.0
        n = len(vtx)
        vtx += [[at(x0), at(y0), z], [at(x1), at(y0), z], [at(x1), at(y1), z], [at(x0), at(y1), z]]
        tri += [[n, n + 1, n + 2], [n, n + 2, n + 3]]
    n2w = np.diag([*flip, 1.0]).astype(np.float32)
    want = _cast_equals_oracle(gpu, oracle, np.array(tri, np.uint32), np.array(vtx, np.float32),
                               n2w, w, w)
    assert (want != 0xFFFFFFFF).sum() > 100


def test_rays_without_direction(gpu, oracle):
    """A camera that maps both NDC planes to one gives rays of length zero,
    which take the general slab test."""
    rng = np.random.default_rng(3)
    vtx = rng.uniform(-1, 1, (60, 3)).astype(np.float32)
    tri = np.arange(60, dtype=np.uint32).reshape(20, 3)
    n2w = np.diag([1.0, 1.0, 0.0, 1.0]).astype(np.float32)
    _cast_equals_oracle(gpu, oracle, tri, vtx, n2w, 16, 16)


# in turn: rays and boxes, only the rays, only the boxes beyond what the regular
# slab test serves; and the mesh's own boxes
@pytest.mark.parametrize("length,far", [(2e-25, 1e20), (2e-25, 1e15), (1e-19, 1e20), (2e-25, 0)])
def test_box_beyond_the_range_of_t(gpu, oracle, length, far):
    """Rays so short that a box's planes lie at t = +inf, beside a parallel axis
    whose slab they miss, in a caller's own boxes: the general test misses such
    a box, whatever the triangles in it."""
    size = 1e13
    rng = np.random.default_rng(5)
    tri, vtx = [], []
    for k in range(40):
        x, y, z = *rng.uniform(-size, size, 2), -1.0 - k
        tri.append([3 * k, 3 * k + 1, 3 * k + 2])
        vtx += [[x - size, y - size, z], [x + size, y - size, z], [x, y + size, z]]
    tri, vtx = np.array(tri, np.uint32), np.array(vtx, np.float32)
    bn, aabb = oracle.build_trimesh3(tri, vtx)
    n2w = np.diag([2 * size, 2 * size, 0.5 * length, 1.0]).astype(np.float32)
    if far:  # all leaves but every fourth
        leaf = np.flatnonzero(bn[:, 2] == 0xFFFFFFFF)
        aabb[leaf[np.arange(len(leaf)) % 4 != 0]] = np.array(
            [3 * size, aabb[0, 1], -2 * far, 4 * size, aabb[0, 4], -far], np.float32)
    dev = [torch.from_numpy(a).to(gpu) for a in (tri, vtx, bn, aabb, n2w)]
    pix, t = Pix2Tri.by_raycasting_with_coeff(*dev, (24, 24))
    want, want_t, _ = oracle.pix2tri(tri, vtx, bn, aabb, n2w.T.reshape(-1), 24, 24, num_threads=4)
    assert np.array_equal(pix.cpu().numpy(), want)
    assert np.array_equal(t.cpu().numpy().view(np.uint32), want_t.view(np.uint32))
    assert 200 < (want != 0xFFFFFFFF).sum() < 576 and _lib.device_errors() == 0


def test_packed_pipeline_holds_one_cast_workspace(gpu):
    """A pipeline that casts from packed buffers keeps the workspace of that cast
    and not the unpacked cast's as well."""
    b = primitives.batch_meshes(4, seed=1, tri_range=(32, 200), pix_range=(500 ** 2, 600 ** 2))
    g = lambda a: torch.from_numpy(a).to(gpu)
    tri, vtx = g(b["tri2vtx"]), g(b["vtx2xyz"])
    need = _lib.lib().dmsh_cast_requests_workspace_bytes(4, int(b["mesh2pix"][-1]))
    assert need > 100 << 20
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated(gpu)
    p = Batched.Pipeline(b["mesh2tri"], b["mesh2vtx"], tri, vtx, b["mesh2pix"], b["mesh2width"],
                         torch.from_numpy(b["ndc2world"]), packed=True)
    assert torch.cuda.memory_allocated(gpu) - before < 1.5 * need
    p.run()
    loop = Batched.PerMeshLoop(p)
    loop.build()
    loop.cast()
    assert torch.equal(p.pix2tri.view(torch.int32), loop.pix2tri.view(torch.int32))
    assert torch.equal(p.pix2t.view(torch.int32), loop.pix2t.view(torch.int32))
    assert _lib.device_errors() == 0
