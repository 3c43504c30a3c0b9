"""Calls whose workspace is smaller than the preferred plan's: they run in the plan that finds room, against the oracle element by
element, and leave a zeroed header zero."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import _assert_every_element, _dev, _say

pytestmark = pytest.mark.gpu

MIB = 1 << 20


# bytes of a caller's workspace, header zeroed or not; None: the fixed array
@pytest.mark.parametrize("room,zeroed,m,n,k,name", [
    (0, False, 49, 7168, 2304, "tile64x64_k1"), (0, False, 621, 768, 2816, "tile64x64_k1"), (0, True, 6006, 96, 3968, "tile64x64_k1"),
    (0, False, 16, 6096, 2432, "_k1"), (32 * MIB, True, 833, 1536, 7168, "tile128x128_k2f"), (32 * MIB, True, 740, 1117, 4864, "padded_"),
    (None, True, 833, 1536, 7168, "tile128x128_k2f"), (None, True, 2805, 576, 7168, ""), (None, True, 345, 4608, 7168, "tile128x128_k2f")])
def test_the_plan_that_finds_room(pkg, room, zeroed, m, n, k, name):
    import torch
    st = torch.cuda.current_stream().cuda_stream
    a, b, sa, sb = oracle.make_inputs(m, n, k, 5100 + m + n + k, 0.5, 30.0)
    dev = _dev(a, b, sa, sb)
    dc = torch.full((m + 16, n), 0x7FC1, dtype=torch.int32, device="cuda").to(torch.int16)
    _say(f"[gpu case] room {room} zeroed {zeroed} m={m} n={n} k={k}")
    if room is None:
        pkg.gemm_noalloc(*dev, dc, m, n, k, st)
    else:
        ws = torch.zeros(max(room, 1), dtype=torch.uint8, device="cuda")
        opt = pkg.Options(flags=pkg.FLAG_WORKSPACE_ZEROED if zeroed else 0)
        for _ in range(2):
            pkg.gemm_ex(*dev, dc, m, n, k, opt, ws if room else None, room, st)
    torch.cuda.synchronize()
    assert name in pkg.last_kernel(), pkg.last_kernel()
    if room and zeroed:
        assert int(ws[:pkg.WORKSPACE_HEADER_BYTES].count_nonzero()) == 0, "header not back to zero"
    got = dc.cpu().numpy().view(np.uint16)
    assert (got[m:] == 0x7FC1).all(), "rows beyond m written"
    _assert_every_element(got[:m], a, b, sa, sb, m, n, k, f"{pkg.last_kernel()} {m}x{n}x{k}")
