"""Tall groups in one launch, with a tile per workgroup and in 128x256 tiles: both tile shapes, rows on and off the 16-row grid, with and without K
splits, against the oracle element by element and bit for bit against the groups one by one; and the launches that dispatch
makes of them."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import _assert_every_element, _dev, _run, _say

pytestmark = pytest.mark.gpu


def _call(pkg, ms, n, k, opt, ws_bytes=None, times=1):
    import torch
    st = torch.cuda.current_stream().cuda_stream
    host = [oracle.make_inputs(m, n, k, 4100 + 7 * g + m + n + k, 0.5, 30.0) for g, m in enumerate(ms)]
    dev = [_dev(*h) for h in host]
    outs = [torch.full((m + 16, n), 0x7FC1, dtype=torch.int32, device="cuda").to(torch.int16) for m in ms]
    ws = torch.zeros(pkg.grouped_workspace_bytes(ms, n, k) if ws_bytes is None else ws_bytes, dtype=torch.uint8, device="cuda")
    _say(f"[gpu case] grouped, a tile per workgroup ms={ms} n={n} k={k} variant={opt.tile_variant} ksplit={opt.ksplit}")
    for _ in range(times):   # what a launch left in the mailbox, the next one would take for its own
        pkg.gemm_grouped_ex(*[[d[i] for d in dev] for i in range(4)], outs, ms, n, k, opt, ws, ws.numel(), st)
    torch.cuda.synchronize()
    if ws.numel() >= pkg.WORKSPACE_HEADER_BYTES:
        assert int(ws[:pkg.WORKSPACE_HEADER_BYTES].count_nonzero()) == 0, "header not back to zero"
    got = []
    for m, o in zip(ms, outs):
        o = o.cpu().numpy().view(np.uint16)
        assert (o[m:] == 0x7FC1).all(), "rows beyond m written"
        got.append(o[:m])
    return host, got, pkg.last_kernel()


# row counts: one less, one more and a whole number of tiles and of 16 rows, the fewest that the form takes; n: ends within a tile;
# K blocks of a split: one, two, odd, more than the ring of four holds; 64 groups: the last lane looks its tile up
@pytest.mark.parametrize("variant,ksplit,ms,n,k", [
    (4, 1, [65, 16, 127, 128, 129, 300], 272, 128), (4, 1, [80, 64, 208], 320, 640), (4, 2, [65, 17, 130], 336, 256),
    (4, 3, [80, 144], 528, 1152), (4, 8, [95, 66, 191], 256, 2048), (4, 5, [257, 31], 304, 3328), (4, 1, [66 + g for g in range(64)], 256, 384),
    (2, 1, [65, 16, 127, 128, 129, 300], 272, 128), (2, 1, [80, 256, 400], 384, 256), (2, 2, [129, 255, 31], 400, 512),
    (2, 3, [144, 128, 272], 256, 1920), (2, 2, [333, 65], 640, 3840), (2, 3, [70 + 3 * g for g in range(20)], 288, 896)])
def test_every_form(pkg, variant, ksplit, ms, n, k):
    opt = pkg.Options(tile_variant=variant, ksplit=ksplit, persistent=0, flags=pkg.FLAG_WORKSPACE_ZEROED)
    host, got, name = _call(pkg, ms, n, k, opt, times=2)
    assert name == f"{'tile64x64' if variant == 4 else 'tile128x128'}_k{ksplit}{'f' if ksplit > 1 else ''}_grouped{len(ms)}", name
    for g, (h, m) in enumerate(zip(host, ms)):
        _assert_every_element(got[g], *h, m, n, k, f"{name} group {g}")
    for g in (0, len(ms) // 2, len(ms) - 1):
        if ms[g] <= 64:   # alone, a batch for the decode kernels
            continue
        a, b, sa, sb = host[g]
        one, single = _run(pkg, a, b, sa, sb, ms[g], n, k, kernel=0, variant=variant, ksplit=ksplit, persistent=0)
        assert np.array_equal(got[g], one), f"{name} group {g} differs from {single}"


@pytest.mark.parametrize("ms,n,k,splits", [([113, 194], 7168, 2048, False), ([299, 81, 66, 130, 75], 544, 256, False), ([151, 246, 201], 448, 5632, True),
                                           ([80, 96, 256, 112], 512, 2944, True), ([67 + 5 * g for g in range(9)], 576, 7168, True), ([67 + 5 * g for g in range(22)], 576, 7168, False)])
def test_automatic_dispatch(pkg, ms, n, k, splits):
    """with the splits where the workspace's header is there and zeroed, else unsplit or as before"""
    opt = pkg.Options(flags=pkg.FLAG_WORKSPACE_ZEROED)
    host, got, name = _call(pkg, ms, n, k, opt, times=3)
    assert name.startswith("tile") and name.endswith(f"_grouped{len(ms)}") and ("f_" in name) == splits, name
    for g, (h, m) in enumerate(zip(host, ms)):
        _assert_every_element(got[g], *h, m, n, k, f"{name} group {g}")
    for flags, ws_bytes in ((0, None), (pkg.FLAG_WORKSPACE_ZEROED, 256)):
        try:
            host, again, name = _call(pkg, ms, n, k, pkg.Options(flags=flags), ws_bytes)
        except pkg.Fp8GemmError as e:   # a plan that needs room for the partial sums of a single group
            assert ws_bytes and "workspace" in str(e), e
            continue
        assert "f_grouped" not in name, name
        for g, (h, m) in enumerate(zip(host, ms)):
            _assert_every_element(again[g], *h, m, n, k, f"{name} group {g}")


# whole rounds; halves of a last round that would leave a quarter of the workgroups or less, or half of them, with a tile; columns
# that end in either half of a tile, rows on and off the grid, the fewest and the most that a group of one tile has
@pytest.mark.parametrize("ms,n,k", [([65 + 7 * g for g in range(9)], 7168, 384), ([128] * 8 + [16], 7216, 2048), ([72 + g for g in range(12)], 7168, 1024),
                                    ([80] * 12 + [128], 6640, 1152), ([127] * 20, 2576, 896)])
def test_groups_of_one_128x256_tile_row(pkg, ms, n, k):
    host, got, name = _call(pkg, ms, n, k, pkg.Options(persistent=1))
    assert name.endswith(f"tile128x256_k1_grouped{len(ms)}"), name
    _, general, pinned = _call(pkg, ms, n, k, pkg.Options(tile_variant=6))
    assert pinned.endswith(f"tile256x256_k1_grouped{len(ms)}"), pinned
    for g, m in enumerate(ms):
        assert np.array_equal(got[g], general[g]), f"group {g}: {name} and {pinned} differ"
        if g in (0, len(ms) - 1):
            _assert_every_element(got[g], *host[g], m, n, k, f"{name} group {g}")


@pytest.mark.parametrize("ms,n,k,name", [([67, 83, 99], 528, 3840, "f_grouped3"), ([90] * 12, 6640, 1152, "tile128x256_k1_grouped12")])
def test_in_a_graph(pkg, ms, n, k, name):
    """every replay, eager work in between, has the eager result"""
    import torch
    dev = [_dev(*oracle.make_inputs(m, n, k, 4700 + g + m, 0.5, 30.0)) for g, m in enumerate(ms)]
    outs = [torch.zeros((m, n), dtype=torch.bfloat16, device="cuda") for m in ms]
    ws = torch.zeros(pkg.grouped_workspace_bytes(ms, n, k), dtype=torch.uint8, device="cuda")
    opt = pkg.Options(persistent=1 if "256" in name else -1, flags=pkg.FLAG_WORKSPACE_ZEROED)

    def call():
        pkg.gemm_grouped_ex(*[[d[i] for d in dev] for i in range(4)], outs, ms, n, k, opt, ws, ws.numel(),
                            torch.cuda.current_stream().cuda_stream)
    _say(f"[gpu case] grouped in a graph ms={ms} n={n} k={k}")
    call()
    torch.cuda.synchronize()
    assert pkg.last_kernel().endswith(name), pkg.last_kernel()
    want = [o.clone() for o in outs]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(4):
        for o in outs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, w) for o, w in zip(outs, want))
        call()


@pytest.mark.parametrize("ms,n,k", [([80 + 16 * (g % 3) for g in range(9)], 576, 7168), ([80, 96, 256, 112], 512, 1920)])
def test_groups_on_the_grid_leave_the_process_wide_workspace_alone(pkg, ms, n, k):
    """what calls on two streams at once would share: split in a workspace of the call's own only"""
    import torch
    _, _, name = _call(pkg, ms, n, k, pkg.Options(flags=pkg.FLAG_WORKSPACE_ZEROED))
    assert "f_grouped" in name, name
    host = [oracle.make_inputs(m, n, k, 4900 + g + m, 0.5, 30.0) for g, m in enumerate(ms)]
    dev = [_dev(*h) for h in host]
    outs = [torch.zeros((m, n), dtype=torch.bfloat16, device="cuda") for m in ms]
    _say(f"[gpu case] grouped on the grid, process-wide workspace ms={ms} n={n} k={k}")
    pkg.gemm_grouped(*[[d[i] for d in dev] for i in range(4)], outs, ms, n, k, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    name = pkg.last_kernel()
    assert name.endswith(f"_grouped{len(ms)}") and "f_" not in name, name
    for g, (h, m) in enumerate(zip(host, ms)):
        _assert_every_element(outs[g].view(torch.int16).cpu().numpy().view(np.uint16), *h, m, n, k, f"{name} group {g}")
