"""GPU: argsort on either side of the lines between the tiles of its digit passes,
with the tiles that the rule takes and with each kind of tile forced."""

import pytest
import torch

from del_msh_dlpack import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [0, 1, 2])
@pytest.mark.parametrize("n", [3 << 19, (3 << 19) + 1, 1 << 21, (1 << 21) + 1, 1 << 22,
                               (1 << 22) + 1, (1 << 23) - 8192, (1 << 23) - 8191])
@pytest.mark.parametrize("bits", [7, 30, 63])
def test_argsort_at_the_lines(gpu, wide, n, bits):
    L = _lib.lib()
    g = torch.Generator(device=gpu).manual_seed(n + bits)
    u64 = bits > 32
    keys = torch.randint(0, 2 ** min(bits, 62), (n,), generator=g, device=gpu)
    keys[: n // 4] = keys[n // 2: n // 2 + n // 4]  # equal keys far apart
    want, order = torch.sort(keys, stable=True)
    dtype = torch.int64 if u64 else torch.int32
    k, idx = keys.to(dtype), torch.empty(n, dtype=torch.int32, device=gpu)
    ws = _lib.workspace(L.dmsh_argsort_workspace_bytes(n, 8 if u64 else 4), gpu)
    old = L.dmsh_get_tuning(b"sort.wide_tiles")
    try:
        assert L.dmsh_set_tuning(b"sort.wide_tiles", wide) == 0
        argsort = L.dmsh_argsort_u64 if u64 else L.dmsh_argsort_u32
        assert argsort(_lib.stream_of(gpu), n, k.data_ptr(), idx.data_ptr(), bits, ws.data_ptr(),
                       ws.numel()) == 0
    finally:
        L.dmsh_set_tuning(b"sort.wide_tiles", old)
    assert torch.equal(k, want.to(dtype)) and torch.equal(idx, order.to(torch.int32))
    assert _lib.device_errors() == 0
