"""Decode launches whose B is read past the caches: every form of the kernels has instances of its own for that.  What a
column of C holds does not depend on the columns beside it: the same problem in pieces of fewer columns, whose B is small
enough to be kept, has the same bits."""
import pytest

pytestmark = pytest.mark.gpu

PIECE = 11_000_000   # bytes of B that are kept in the caches whatever the launch


def _codes(gen, *shape):
    import torch
    x = torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)
    return torch.where((x & 0x7F) == 0x7F, x & 0x80, x)   # no NaN


def _problem(gen, m, n, k):
    import torch
    scales = lambda *shape: torch.rand(shape, device="cuda", generator=gen) + 0.5
    return _codes(gen, k, m), _codes(gen, k, n), scales(k // 128, m), scales(k // 128, n // 128)


def _single(pkg, a, b, sa, sb, c, m, n, k, variant, ksplit):
    import torch
    pkg.select(pkg.KERNEL_SKINNY)
    pkg.force_config(variant, ksplit)
    try:
        pkg.gemm(a, b, sa, sb, c, m, n, k, torch.cuda.current_stream().cuda_stream)
        assert pkg.last_kernel() == f"decode{128 * variant}_k{ksplit}", pkg.last_kernel()
    finally:
        pkg.force_config(-1, 0)
        pkg.select(0)


def _in_pieces(pkg, a, b, sa, sb, m, n, k, ksplit):
    import torch
    out = torch.empty((m, n), dtype=torch.int16, device="cuda")
    step = max(128, PIECE // k // 128 * 128)
    for at in range(0, n, step):
        cols = min(step, n - at)
        c = torch.empty((m, cols), dtype=torch.int16, device="cuda")
        _single(pkg, a, b[:, at:at + cols].contiguous(), sa, sb[:, at // 128:(at + cols) // 128].contiguous(), c, m, cols, k, 1, ksplit)
        out[:, at:at + cols] = c
    return out


@pytest.mark.parametrize("variant,ksplit,n,k,rows,offset", [
    (1, 4, 7168, 2048, (1, 8, 15, 16), 0),         # a single row tile over a small B; two stages to a barrier
    (1, 6, 4608, 7168, (24, 31, 32), 0),           # two row tiles
    (1, 4, 8192, 4096, (40, 47, 48, 56, 63, 64), 0),
    (1, 3, 16384, 7168, (8, 15, 16, 24, 31, 32), 0),   # more workgroups than CUs: one stage to a barrier
    (1, 2, 16384, 7168, (16, 32), 0),              # 28 K blocks each: rows on the grid in the instances that spread them
    (1, 1, 28672, 6784, (16, 24, 47, 64), 0),      # unsplit
    (2, 1, 49152, 2432, (16, 24, 31, 47, 56, 64), 0),  # strips of 256 columns, one round
    (2, 3, 18432, 7168, (8, 15, 16, 32), 0),       # ... and split
    (1, 1, 65536, 1792, (16, 32, 48, 64), 0),      # streaming, strips of 256 columns
    (1, 1, 65536, 1792, (16, 32, 48, 64), 4),      # ... C on an 8-byte boundary
    (1, 1, 33024, 5888, (16, 32, 48, 64), 0),      # streaming, strips of 128 columns
    (1, 1, 33024, 5888, (16, 64), 4),
])
def test_single_problem(pkg, variant, ksplit, n, k, rows, offset):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n + k + ksplit)
    for m in rows:
        a, b, sa, sb = _problem(gen, m, n, k)
        flat = torch.full((offset + m * n + 64,), 0x7FC1, dtype=torch.int16, device="cuda")
        got = flat[offset:offset + m * n].view(m, n)
        print(f"[gpu case] B past the caches: {m}x{n}x{k} variant={variant} ksplit={ksplit} c+{offset}", flush=True)
        _single(pkg, a, b, sa, sb, got, m, n, k, variant, ksplit)
        want = _in_pieces(pkg, a, b, sa, sb, m, n, k, ksplit)
        torch.cuda.synchronize()
        assert torch.equal(got, want), m
        assert (flat[:offset] == 0x7FC1).all() and (flat[offset + m * n:] == 0x7FC1).all(), "written beside C"
    pkg.release()


@pytest.mark.parametrize("ms,n,k,ksplit", [
    ([16] * 64, 1024, 256, 1),                 # streaming
    ([16, 64] * 32, 1024, 256, 1),             # ... with up to four row tiles
    ([5, 16] * 5, 3072, 512, 1),               # rows off the grid: two stages to a barrier, and one
    ([5, 16] * 4, 4096, 384, 1),
    ([33, 7] * 4, 4096, 512, 1),
    ([33, 7] * 4, 4096, 384, 1),
    ([16, 32] * 4, 4096, 512, 1),              # rows on the grid
    ([48, 16] * 4, 4096, 512, 1),
    ([16] * 9, 4096, 512, 1),
    ([48] * 9, 4096, 512, 1),
    ([16, 7] + [32], 3072, 2048, 4),           # 72 strips, 288 workgroups
    ([16] * 64, 2048, 1536, 2),                # 2048 workgroups: the ring of three
])
def test_grouped(pkg, ms, n, k, ksplit):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n + k + len(ms))
    groups = [_problem(gen, m, n, k) for m in ms]
    got = [torch.full((m + 1, n), 0x7FC1, dtype=torch.int16, device="cuda") for m in ms]   # one guard row
    print(f"[gpu case] B past the caches: grouped {ms} {n}x{k} ksplit={ksplit}", flush=True)
    pkg.force_config(-1, ksplit)
    try:
        pkg.gemm_grouped(*[[x[i] for x in groups] for i in range(4)], got, ms, n, k, torch.cuda.current_stream().cuda_stream)
        assert pkg.last_kernel() == f"decode128_k{ksplit}_grouped{len(ms)}", pkg.last_kernel()
    finally:
        pkg.force_config(-1, 0)
    for g, m in enumerate(ms):
        want = _in_pieces(pkg, *groups[g], m, n, k, ksplit)
        torch.cuda.synchronize()
        assert torch.equal(got[g][:m], want), g
        assert (got[g][m] == 0x7FC1).all(), "rows beyond m written"
    pkg.release()
