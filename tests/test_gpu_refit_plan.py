"""GPU: the plan that a standalone refit keeps in its workspace is used only while
it is whole, whatever the memory was used for since it was made."""

import threading

import numpy as np
import pytest
import torch

import del_msh_dlpack.TriMesh3.torch as TriMesh3
from del_msh_dlpack import _lib, primitives

pytestmark = pytest.mark.gpu


def G(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def same_bits(t, want):
    return np.array_equal(t.cpu().numpy().view(np.uint32), want.view(np.uint32))


def refit(gpu, pts, bn, ws):
    L = _lib.lib()
    aabb = torch.full((bn.shape[0], 6), float("nan"), device=gpu)
    t_pts, t_bn = G(pts, gpu), G(bn, gpu)
    _lib.check(L.dmsh_bvhnode2aabb_points(
        _lib.stream_of(gpu), _lib.ptr(aabb), bn.shape[0], _lib.ptr(t_bn), pts.shape[0],
        _lib.ptr(t_pts), _lib.ptr(ws), ws.numel()), "dmsh_bvhnode2aabb_points")
    return aabb


def cloud(oracle, n):
    pts = np.random.default_rng(n).random((n, 3), dtype=np.float32)
    return pts, oracle.build_points(pts, morton_bits=63)[0]


def test_trees_of_several_sizes_share_a_workspace(gpu, oracle):
    # the parts of a workspace lie where the size puts them: 5000 leaves write
    # over the lists of 2 leaves and not over their stamp, 70 000 over those of
    # 5000, and so on down and up again
    clouds = {n: cloud(oracle, n) for n in (2, 3, 1025, 5000, 64_000, 70_000, 300_000)}
    want = {n: oracle.refit_points(bn, pts) for n, (pts, bn) in clouds.items()}
    ws = torch.full((_lib.lib().dmsh_refit_workspace_bytes(300_000),), 0xA5, dtype=torch.uint8,
                    device=gpu)
    order = [2, 5000, 2, 3, 70_000, 5000, 2, 300_000, 70_000, 3, 1025, 5000, 300_000, 1025, 70_000]
    order += list(np.random.default_rng(1).choice(list(clouds), 25))
    for step, n in enumerate(order):
        assert same_bits(refit(gpu, *clouds[n], ws), want[n]), (step, n)
    assert _lib.device_errors() == 0


def test_meshes_of_several_sizes_by_the_module(gpu, oracle):
    meshes = {}
    for n in (1, 50, 150):
        tri, vtx = (np.arange(6, dtype=np.uint32).reshape(2, 3),
                    np.random.default_rng(3).random((6, 3), dtype=np.float32)) if n == 1 else \
            primitives.torus_zup(0.7, 0.3, n, n)
        bn = oracle.build_trimesh3(tri, vtx)[0]
        meshes[n] = tri, vtx, bn, oracle.refit_trimesh3(bn, tri, vtx, 0.0)
    # the largest first: the workspace that the module keeps does not grow after it
    for n in (150, 1, 50, 1, 150, 50, 1, 150):
        tri, vtx, bn, want = meshes[n]
        got = TriMesh3.make_bvhnode2aabb_from_bvhnodes(G(tri, gpu), G(vtx, gpu), G(bn, gpu))
        assert same_bits(got, want), n
    assert _lib.device_errors() == 0


@pytest.mark.parametrize("part", ["treelets", "top_list", "node2slot", "count", "failed"])
def test_a_plan_that_was_written_over_is_made_again(gpu, oracle, part):
    """Two entries of a list exchanged (or a count changed) behind the stamp's
    back: the next call must not keep the plan, and the one after must."""
    n = 100_000
    nb, (pts, bn) = n - 1, cloud(oracle, n)
    if part == "failed":  # leaves 3 and n - 5 exchanged: not an LBVH's leaf ranges
        bn = bn.copy()
        r1, r2 = nb + 3, nb + n - 5
        p1, p2 = int(bn[r1, 0]), int(bn[r2, 0])
        assert p1 != p2
        bn[p1, 1:] = np.where(bn[p1, 1:] == r1, r2, bn[p1, 1:])
        bn[p2, 1:] = np.where(bn[p2, 1:] == r2, r1, bn[p2, 1:])
        bn[[r1, r2]] = bn[[r2, r1]]
    want = oracle.refit_points(bn, pts)
    ws = torch.zeros(_lib.lib().dmsh_refit_workspace_bytes(n), dtype=torch.uint8, device=gpu)
    words = ws[: ws.numel() // 4 * 4].view(torch.int32)
    # word offsets: four arrays of n - 1 words, the counters, the lists, each on 256 bytes
    slot = (nb + 63) // 64 * 64
    node2slot, counters = 3 * slot, 4 * slot
    treelets = counters + 64
    top_list = treelets + (4 * n + 63) // 64 * 64

    def kept():
        assert same_bits(refit(gpu, pts, bn, ws), want)
        assert _lib.device_errors() == 0
        return int(words[counters + 4]) == 0

    assert not kept()
    assert kept() == (part != "failed")
    nt, tc = int(words[counters]), int(words[counters + 1])
    assert nt > 2 and tc > 2 or part == "failed"
    if part == "count":
        words[counters] = nt - 1
    elif part == "failed":
        words[counters: counters + 4] = 0
    else:
        if part == "node2slot":
            a, b = (node2slot + int(words[top_list + 4 * e]) for e in (0, 1))
            a, b = slice(a, a + 1), slice(b, b + 1)
        else:
            base = treelets if part == "treelets" else top_list
            a, b = slice(base, base + 4), slice(base + 4, base + 8)
        x, y = words[a].clone(), words[b].clone()
        words[a], words[b] = y, x
    assert not kept()
    assert kept() == (part != "failed")


def test_a_captured_refit_outlives_the_kept_workspace(gpu, oracle):
    """A graph holds its workspace's address: later refits of larger trees, which
    replace the kept workspace, must not take it away from the graph, nor the
    replays write into what the allocator made of it."""
    rng = np.random.default_rng(5)
    tri, vtx = primitives.torus_zup(0.7, 0.3, 40, 30)
    bn = oracle.build_trimesh3(tri, vtx)[0]
    t_tri, t_vtx, t_bn = G(tri, gpu), G(vtx, gpu), G(bn, gpu)
    stream = torch.cuda.Stream(gpu)
    with torch.cuda.stream(stream):
        TriMesh3.make_bvhnode2aabb_from_bvhnodes(t_tri, t_vtx, t_bn)
        torch.cuda.synchronize()
        key = ("dmsh_bvhnode2aabb_trimesh3", gpu.index or 0, stream.cuda_stream)
        kept = _lib._KEPT[key].ws
        before = kept.clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            aabb = TriMesh3.make_bvhnode2aabb_from_bvhnodes(t_tri, t_vtx, t_bn)
        assert _lib._KEPT[key].ws is kept
        for step, n in enumerate((0, 60, 90, 120)):
            if n:  # a larger tree: a larger kept workspace, and new tensors where the old one was
                btri, bvtx = primitives.torus_zup(0.7, 0.3, n, n)
                bbn = oracle.build_trimesh3(btri, bvtx)[0]
                got = TriMesh3.make_bvhnode2aabb_from_bvhnodes(G(btri, gpu), G(bvtx, gpu),
                                                               G(bbn, gpu))
                assert same_bits(got, oracle.refit_trimesh3(bbn, btri, bvtx, 0.0)), n
                kept = before = None
            fill = [torch.full((1 << 18,), 7, dtype=torch.int32, device=gpu) for _ in range(8)]
            moved = (vtx + rng.normal(size=vtx.shape) * 0.01).astype(np.float32)
            t_vtx.copy_(G(moved, gpu))
            aabb.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert same_bits(aabb, oracle.refit_trimesh3(bn, tri, moved, 0.0)), step
            assert all(bool((f == 7).all()) for f in fill), step
            if kept is not None:
                assert torch.equal(kept, before)  # the replay ran in a workspace of its own
    assert _lib.device_errors() == 0


def test_threads_share_a_stream(gpu, oracle):
    """Refits of two trees by two threads on one stream share its workspace: the
    launches of one call must not come between those of the other."""
    errors = []

    def work(n):
        try:
            tri, vtx = primitives.torus_zup(0.7, 0.3, n, n)
            bn = oracle.build_trimesh3(tri, vtx)[0]
            want = G(oracle.refit_trimesh3(bn, tri, vtx, 0.0), gpu)
            t_tri, t_vtx, t_bn = G(tri, gpu), G(vtx, gpu), G(bn, gpu)
            wrong = torch.zeros((), dtype=torch.int64, device=gpu)
            for _ in range(300):
                wrong += (TriMesh3.make_bvhnode2aabb_from_bvhnodes(t_tri, t_vtx, t_bn)
                          != want).any()
            if int(wrong):
                errors.append((n, int(wrong)))
        except Exception as e:  # pylint: disable=broad-except
            errors.append((n, e))

    threads = [threading.Thread(target=work, args=(n,)) for n in (40, 90)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors
    assert _lib.device_errors() == 0
