"""K splits added inside the tile kernels with four multiplying waves, whose copy waves gather half of the patches: every
number of senders around a trip, cut tiles, rows off the grid, bit for bit what the reduction kernel adds; zeros left behind."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import _assert_every_element, _dev, _run, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant,ksplit,m,n,k", [
    *((4, s, 80, 144, 128 * (2 * s - 1)) for s in (2, 3, 4, 5, 6, 7, 8)),   # the last split a block short
    (4, 4, 64, 64, 512), (4, 3, 77, 208, 1024), (4, 8, 117, 80, 2048),              # one block each; rows off the grid
    (2, 2, 144, 208, 4096), (2, 3, 256, 144, 6016), (2, 4, 128, 128, 8192), (2, 2, 400, 272, 3968)])
def test_splits_added_by_eight_waves(pkg, variant, ksplit, m, n, k):
    import torch
    a, b, sa, sb = oracle.make_inputs(m, n, k, 3100 + m + n + k, 0.5, 30.0)
    want, name = _run(pkg, a, b, sa, sb, m, n, k, kernel=pkg.KERNEL_SPLITK, variant=variant, ksplit=ksplit, fused=0)
    _assert_every_element(want, a, b, sa, sb, m, n, k, name)
    da, db, dsa, dsb = _dev(a, b, sa, sb)
    st = torch.cuda.current_stream().cuda_stream
    pkg.set_fused_reduction(1)
    try:
        opt = pkg.Options(kernel=pkg.KERNEL_SPLITK, tile_variant=variant, ksplit=ksplit, flags=pkg.FLAG_WORKSPACE_ZEROED)
        ws = torch.zeros(max(pkg.workspace_bytes_ex(m, n, k, opt), pkg.WORKSPACE_HEADER_BYTES), dtype=torch.uint8, device="cuda")
        dc = torch.full((m + 16, n), 0x7FC1, dtype=torch.int32, device="cuda").to(torch.int16)
        _say(f"[gpu case] splits added inside: {name} {m}x{n}x{k}")
        for _ in range(3):
            pkg.gemm_ex(da, db, dsa, dsb, dc, m, n, k, opt, ws, ws.numel(), st)
        torch.cuda.synchronize()
    finally:
        pkg.set_fused_reduction(-1)
    assert pkg.last_kernel() == name + "f", pkg.last_kernel()
    assert np.array_equal(want, dc[:m].cpu().numpy().view(np.uint16)), f"{name}: differs from the reduction kernel's result"
    assert (dc[m:].cpu().numpy().view(np.uint16) == 0x7FC1).all(), "rows beyond m written"
    assert int(ws[:pkg.WORKSPACE_HEADER_BYTES].count_nonzero()) == 0, "header not back to zero"
