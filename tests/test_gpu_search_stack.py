"""GPU: point location where the walk's stack fills up and where the whole tree
is walked in vain, and interpolation of one to five values a vertex, against the
oracle."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib, primitives
import del_msh_dlpack.PolyhedronMesh.torch as PolyhedronMesh

pytestmark = pytest.mark.gpu


# a chain of equal codes: 32 frames in LDS, deeper walks climb
@pytest.mark.parametrize("copies", [1, 2, 31, 32, 33, 34, 35, 70, 200])
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("vdim", [1, 2, 3, 5])
def test_deep_walks(gpu, oracle, copies, flip, vdim):
    tet = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], np.float32)
    other = (1.0 - tet).astype(np.float32)  # fills the opposite corner of the box
    x = np.concatenate([tet, other, tet + 4.0]).astype(np.float32)
    elems = [[0, 1, 2, 3]] * copies + [[4, 5, 6, 7], [8, 9, 10, 11]]
    if flip:
        elems = elems[::-1]
    off = np.arange(0, 4 * len(elems) + 1, 4, dtype=np.uint32)
    iv = np.asarray(elems, np.uint32).reshape(-1)
    rng = np.random.default_rng(copies)
    q = np.concatenate([rng.uniform(0, 1, (200, 3)), rng.uniform(-1, 6, (100, 3))]).astype(np.float32)
    g = lambda a: torch.from_numpy(a).to(gpu)
    bn, _ = oracle.build_points(oracle.polyhedron_elem2center(off, iv, x))
    aabb = oracle.polyhedron_refit(bn, off, iv, x)
    elem, par = PolyhedronMesh.search_elem_contain_points(g(off), g(iv), g(x), g(bn), g(aabb), g(q))
    want, want_par = oracle.polyhedron_search(off, iv, x, bn, aabb, q)
    assert np.array_equal(elem.cpu().numpy(), want)
    assert np.array_equal(par.cpu().numpy().view(np.uint32), want_par.view(np.uint32))
    assert (want == 0xFFFFFFFF).any() and (want != 0xFFFFFFFF).any()
    val = rng.standard_normal((x.shape[0], vdim)).astype(np.float32)
    got = PolyhedronMesh.interpolate_values_at_points(g(off), g(iv), g(val), elem, par)
    want_val = oracle.polyhedron_interpolate(off, iv, val, want, want_par)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want_val.view(np.uint32))
    assert _lib.device_errors() == 0


def test_arrays_at_a_four_byte_boundary(gpu, oracle):
    """The tree and the points as slices of larger buffers, aligned to their
    elements and to nothing more."""
    off, iv, x = primitives.mixed_hex_grid(4, 4, 4, seed=2)
    rng = np.random.default_rng(0)
    q = rng.uniform(-0.2, 4.2, (500, 3)).astype(np.float32)
    bn, _ = oracle.build_points(oracle.polyhedron_elem2center(off, iv, x))
    aabb = oracle.polyhedron_refit(bn, off, iv, x)

    def shifted(a):
        b = torch.empty(a.size + 1, dtype=torch.from_numpy(a).dtype, device=gpu)[1:].view(a.shape)
        assert b.data_ptr() % 8 == 4 and b.is_contiguous()
        return b.copy_(torch.from_numpy(a))

    elem, par = PolyhedronMesh.search_elem_contain_points(
        *map(shifted, (off, iv, x.astype(np.float32), bn, aabb, q)))
    want, want_par = oracle.polyhedron_search(off, iv, x, bn, aabb, q)
    assert np.array_equal(elem.cpu().numpy(), want)
    assert np.array_equal(par.cpu().numpy().view(np.uint32), want_par.view(np.uint32))
    assert (want != 0xFFFFFFFF).sum() > 300 and _lib.device_errors() == 0


@pytest.mark.parametrize("dims", [(12, 12, 12), (60, 40, 1), (1, 900, 1), (3, 1, 500), (1, 1, 1)])
@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e30, 0.0])
def test_order_of_queries_in_boxes_of_every_shape(gpu, oracle, dims, scale):
    """Queries enough to be put in order: in cubes, plates, rods and a mesh that
    is drawn together in a point, inside, outside and not finite."""
    off, iv, x = primitives.mixed_hex_grid(*dims, seed=3)
    x = (x * scale).astype(np.float32)
    rng = np.random.default_rng(1)
    q = (rng.uniform(-0.1, 1.1, (1000, 3)) * np.array(dims) * scale).astype(np.float32)
    q[::97] = np.nan
    q[::101, 1] = np.inf
    bn, _ = oracle.build_points(oracle.polyhedron_elem2center(off, iv, x))
    aabb = oracle.polyhedron_refit(bn, off, iv, x)
    want, want_par = oracle.polyhedron_search(off, iv, x, bn, aabb, q)
    assert scale != 1.0 or (want != 0xFFFFFFFF).sum() > 300
    which = rng.permutation(np.arange(70000) % 1000)
    elem, par = PolyhedronMesh.search_elem_contain_points(
        *(torch.from_numpy(a).to(gpu) for a in (off, iv, x, bn, aabb, q[which])))
    assert np.array_equal(elem.cpu().numpy(), want[which])
    assert np.array_equal(par.cpu().numpy().view(np.uint32), want_par[which].view(np.uint32))
    assert _lib.device_errors() == 0
