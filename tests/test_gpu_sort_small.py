"""GPU: the argsort by merged LDS chunks at the edges of its chunks and past its
end, against numpy's stable argsort."""

import numpy as np
import pytest
import torch

from del_msh_dlpack import _lib
import del_msh_dlpack.Array1D.torch as Array1D

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 8193, 16384, 16385, 20481, 24576, 24577,
         28672, 28673, 36864, 36865, 40960, 40961, 53248, 53249, 65537,
         98304, 98305]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("bits,key_bits", [(32, 32), (32, 30), (32, 9), (32, 1), (64, 63), (64, 64)])
def test_argsort_small(gpu, n, bits, key_bits):
    rng = np.random.default_rng(n + key_bits)
    dt = np.uint32 if bits == 32 else np.uint64
    top = (1 << key_bits) - 1
    spread = rng.integers(0, top, n, dtype=np.uint64, endpoint=True)
    # runs of equal keys, and keys of all ones next to the padding
    few = rng.choice(np.array([0, 1, top >> 1, top], np.uint64), n)
    for keys in (spread.astype(dt), few.astype(dt)):
        idx, val = Array1D.argsort(torch.from_numpy(keys).to(gpu), key_bits)
        want = np.argsort(keys, kind="stable")
        assert np.array_equal(idx.cpu().numpy(), want.astype(np.uint32))
        assert np.array_equal(val.cpu().numpy(), keys[want])
    assert _lib.device_errors() == 0
