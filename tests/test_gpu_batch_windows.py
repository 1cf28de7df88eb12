"""GPU: batched builds whose meshes' boundaries fall around the batched
kernels' windows (rounds of 256 triangles with more meshes than the window of
four, blocks of 256 nodes over one and many meshes) and whose codes repeat,
against the single-mesh build bit for bit."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib
import del_msh_dlpack.Batched.torch as Batched

pytestmark = pytest.mark.gpu

SIZES = {
    "ones": [1] * 600,
    "small": [0, 3, 60, 64, 65, 2, 1, 0, 0, 5, 31, 32, 33] * 20,
    "edges": [255, 256, 257, 1, 0, 1, 1, 1, 1, 1000, 2, 511, 513, 4096, 7],
    "large": [5000, 3, 12289, 0, 2, 30000],
}


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("codes", ["spread", "repeated"])
def test_batched_build_equals_single_builds(gpu, sizes, codes):
    n = np.array(SIZES[sizes])
    rng = np.random.default_rng(3)
    csr = lambda c: np.concatenate([[0], np.cumsum(c)]).astype(np.uint32)
    v = rng.normal(size=(int(3 * n.sum()), 3)).astype(np.float32)
    if codes == "repeated":
        v = np.round(v)  # centroids on a coarse grid: runs of equal codes
    tri = np.concatenate([np.arange(3 * k, dtype=np.uint32).reshape(-1, 3) for k in n])
    g = lambda a: torch.from_numpy(a).to(gpu)
    p = Batched.Pipeline(csr(n), csr(3 * n), g(tri), g(v))
    p.build()
    single = Batched.PerMeshLoop(p)
    single.build()
    assert single.equals_pipeline()
    assert _lib.device_errors() == 0
