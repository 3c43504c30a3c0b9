"""The decode kernel with 64-column strips, pinned by name: every way its rows of A lie in a stage and every number of row
tiles, at the ends of its ranges, against the oracle element by element; and the plans that dispatch makes with it."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import _assert_every_element, _dev, _run, _say

pytestmark = pytest.mark.gpu

# n: one column patch, a strip, less and more than one, strips dealt out over the XCDs (up to 16) and in pairs (more), an odd
# number of them; K blocks of a split: one, two, odd, more than the ring holds; splits: none, one trip of the hand-over, two
SHAPES = [(16, 128, 1), (64, 256, 1), (80, 384, 3), (576, 7168, 14), (1040, 2048, 16), (1072, 1152, 3), (1536, 2560, 4),
          (272, 3584, 2), (2064, 1280, 1)]


@pytest.mark.parametrize("m", [1, 2, 7, 8, 15, 16, 17, 24, 31, 32, 33, 40, 48, 49, 56, 64])
def test_strips_of_64_columns(pkg, m):
    for n, k, ksplit in SHAPES:
        a, b, sa, sb = oracle.make_inputs(m, n, k, 2100 + m + n + k, 0.5, 30.0)
        got, name = _run(pkg, a, b, sa, sb, m, n, k, kernel=pkg.KERNEL_SKINNY, variant=3, ksplit=ksplit)
        assert name == f"decode64_k{ksplit}", name
        _assert_every_element(got, a, b, sa, sb, m, n, k, f"{name} {m}x{n}x{k}")
        again, _ = _run(pkg, a, b, sa, sb, m, n, k, kernel=pkg.KERNEL_SKINNY, variant=3, ksplit=ksplit)
        assert np.array_equal(got, again), f"{name}: not reproducible"


@pytest.mark.parametrize("m,n,k", [(1, 7168, 256), (1, 512, 7168), (3, 576, 7168), (24, 1536, 7168), (31, 3072, 1536), (40, 576, 7168),
                                   (48, 1536, 7168), (56, 528, 6656)])
def test_automatic_dispatch(pkg, m, n, k):
    """in a caller's workspace, three launches in a row; rows behind C untouched, the header back to zero; a off the 16-byte
    grid, which runs on padded copies, is within the same bounds"""
    import torch
    st = torch.cuda.current_stream().cuda_stream
    a, b, sa, sb = oracle.make_inputs(m, n, k, 2200 + m + n + k, 0.5, 30.0)
    da, db, dsa, dsb = _dev(a, b, sa, sb)
    opt = pkg.Options(flags=pkg.FLAG_WORKSPACE_ZEROED)
    need = pkg.workspace_bytes_ex(m, n, k, opt, any_alignment=True)
    ws = torch.zeros(max(need, 256), dtype=torch.uint8, device="cuda")
    dc = torch.full((m + 16, n), 0x7FC1, dtype=torch.int32, device="cuda").to(torch.int16)
    _say(f"[gpu case] automatic dispatch m={m} n={n} k={k}")
    for _ in range(3):
        pkg.gemm_ex(da, db, dsa, dsb, dc, m, n, k, opt, ws, ws.numel(), st)
    torch.cuda.synchronize()
    name = pkg.last_kernel()
    assert name.startswith("decode64_k"), name
    got = dc[:m].cpu().numpy().view(np.uint16)
    _assert_every_element(got, a, b, sa, sb, m, n, k, name)
    assert (dc[m:].cpu().numpy().view(np.uint16) == 0x7FC1).all(), "rows beyond m written"
    assert int(ws[:pkg.WORKSPACE_HEADER_BYTES].count_nonzero()) == 0, "header not back to zero"
    shifted = torch.zeros(a.size + 16, dtype=torch.uint8, device="cuda")
    shifted[4:4 + a.size] = da.view(torch.uint8).reshape(-1)
    dc.fill_(0x7FC1)
    pkg.gemm_ex(shifted[4:4 + a.size], db, dsa, dsb, dc, m, n, k, opt, ws, ws.numel(), st)
    torch.cuda.synchronize()
    assert pkg.last_kernel().startswith("padded_"), pkg.last_kernel()
    _assert_every_element(dc[:m].cpu().numpy().view(np.uint16), a, b, sa, sb, m, n, k, pkg.last_kernel())
    assert (dc[m:].cpu().numpy().view(np.uint16) == 0x7FC1).all(), "rows beyond m written"


# more splits than any plan has; splits that may not meet in the mailbox; 256 strips x 7 sending splits x 16 KiB of patches, which do
# not fit it
@pytest.mark.parametrize("m,n,k,ksplit,fused", [(16, 512, 4096, 17, -1), (16, 512, 4096, 4, 0), (64, 16384, 2048, 8, -1)])
def test_a_split_that_does_not_exist_is_refused(pkg, m, n, k, ksplit, fused):
    a, b, sa, sb = oracle.make_inputs(m, n, k, 2300)
    with pytest.raises(pkg.Fp8GemmError) as info:
        _run(pkg, a, b, sa, sb, m, n, k, kernel=pkg.KERNEL_SKINNY, variant=3, ksplit=ksplit, fused=fused)
    assert info.value.code == -3


def test_the_most_that_fits_the_mailbox(pkg):
    m, n, k = 64, 16384, 2560
    a, b, sa, sb = oracle.make_inputs(m, n, k, 2301, 0.5, 30.0)
    got, name = _run(pkg, a, b, sa, sb, m, n, k, kernel=pkg.KERNEL_SKINNY, variant=3, ksplit=5)
    assert name == "decode64_k5", name
    _assert_every_element(got, a, b, sa, sb, m, n, k, f"{name} {m}x{n}x{k}")
