"""GPU: smoothing over one, two and more launches (odd and even numbers of
them) equals the same sweeps one launch at a time, bit for bit, on images
smaller and larger than a tile."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib
import del_msh_dlpack.RasterizedEdgeGradient.torch as REG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_iter", [8, 9, 16, 20, 33])  # eight sweeps a launch
@pytest.mark.parametrize("w, h", [(2, 2), (31, 33), (65, 32), (150, 97)])
def test_launches_chain(gpu, num_iter, w, h):
    rng = np.random.default_rng(num_iter + w)
    g = lambda a: torch.from_numpy(a).to(gpu)
    kind = lambda *s: g(rng.choice(5, size=s, p=[0.5, 0.2, 0.1, 0.1, 0.1]).astype(np.uint8))
    ht, vt = kind(h - 1, w), kind(h, w - 1)
    hd, vd = (g(rng.normal(size=t.shape).astype(np.float32)) for t in (ht, vt))
    one_h, one_v = hd.clone(), vd.clone()
    REG.smooth_gradient(ht, vt, num_iter, hd, vd)
    for _ in range(num_iter):
        REG.smooth_gradient(ht, vt, 1, one_h, one_v)
    assert torch.equal(hd.view(torch.int32), one_h.view(torch.int32))
    assert torch.equal(vd.view(torch.int32), one_v.view(torch.int32))
    assert _lib.device_errors() == 0
