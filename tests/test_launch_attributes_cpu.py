"""Which kernels calls launch and what the launches ask for, with stand-ins for the runtime's calls: no device, nothing
runs."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(pkg, tmp_path_factory):
    lib = pkg.lib_path()
    exe = str(tmp_path_factory.mktemp("stand_in") / "stand_in_runtime")
    subprocess.run(["gcc", "-O1", "-Wall", "-rdynamic", os.path.join(HERE, "stand_in_runtime.c"), lib, "-Wl,-rpath," + os.path.dirname(lib),
                    "-Wl,--unresolved-symbols=ignore-in-shared-libs", "-o", exe], check=True)
    return lambda *args: subprocess.run([exe, *map(str, args)], check=True, capture_output=True, text=True, timeout=120).stdout.split()


def test_the_lds_limit_is_raised_once_for_each_kernel(program):
    words = program()
    count = {name: int(value) for name, value in zip(words[::2], words[1::2])}
    assert count["calls"] > 1000 and count["kernels"] > 60, count
    assert count["missing"] == 0 and count["again"] == 0 and count["raised"] >= count["kernels"], count


def reads_past_the_caches(program, m, n, k, split=0, groups=0):
    kernels = [name for name in program(m, n, k, split, groups) if "decode_" in name]
    assert len(kernels) == 1, kernels
    name = subprocess.run(["c++filt", kernels[0]], check=True, capture_output=True, text=True).stdout
    assert ", true>(" in name or ", false>(" in name, name   # ONCE is the last template argument
    return ", true>(" in name


# B that the caches hold from call to call stays there where it comes slower past them: two row tiles over a small B, mid-sized
# ones, unsplit launches of 128-column strips; what does not fit the Infinity Cache is read past it whatever the launch
@pytest.mark.parametrize("m,n,k,past", [(1, 7168, 2048, True), (16, 7168, 2048, True), (24, 7168, 2048, False), (32, 7168, 2048, False),
                                        (24, 4608, 7168, True), (8, 10240, 2048, False), (32, 9216, 3072, False), (16, 7168, 7168, False),
                                        (24, 7168, 2304, False), (16, 28672, 2048, False), (16, 28672, 4096, False), (32, 16384, 7168, True),
                                        (48, 16384, 7168, False), (16, 57344, 2048, True), (48, 65536, 3072, True), (31, 28672, 8192, True),
                                        (16, 7152, 2048, False)])
def test_which_b_is_read_past_the_caches(program, m, n, k, past):
    assert reads_past_the_caches(program, m, n, k) == past


# 72 strips in four splits and 84 in three are launches of more than 200 workgroups, 84 unsplit are not
@pytest.mark.parametrize("groups,m,n,k,split,past", [(3, 16, 3072, 2048, 4, True), (7, 32, 1536, 2048, 3, True), (7, 32, 1536, 2048, 1, False),
                                                     (16, 32, 7168, 2048, 1, True), (2, 16, 1536, 2048, 4, False), (64, 32, 7152, 2048, 1, False)])
def test_grouped_launches_count_their_workgroups(program, groups, m, n, k, split, past):
    assert reads_past_the_caches(program, m, n, k, split, groups) == past


# 128x128 tiles: four waves of 64x64, or eight of 64x32 where the chains are short
@pytest.mark.parametrize("m,n,k,split,waves", [(1392, 720, 1024, 2, 8), (3824, 272, 2176, 2, 8), (1376, 624, 5760, 3, 8),
                                               (2048, 576, 7168, 3, 4), (256, 1024, 4096, 2, 4), (253, 1024, 4096, 2, 8),
                                               (416, 3824, 128, 1, 8), (413, 3824, 128, 1, 8), (416, 3824, 256, 1, 4), (413, 3824, 256, 1, 4),
                                               (1024, 4096, 2048, 4, 4)])   # the last: more than the mailbox holds, a reduction kernel
def test_waves_of_128x128_tiles(program, m, n, k, split, waves):
    names = subprocess.run(["c++filt"], input="\n".join(program(m, n, k, split, 0, 2)), check=True, capture_output=True, text=True).stdout
    assert f"tile_gemm_kernel<128, 128, 2, {waves // 2}, 4, {'true' if split > 1 else 'false'}, {'true' if m % 16 else 'false'}>" in names, names


# 256x192 tiles in a single round: the persistent kernel over more than eight K blocks, also on padded copies
@pytest.mark.parametrize("m,n,k,persistent", [(1424, 7168, 2048, True), (2512, 4608, 7168, True), (3608, 3072, 1536, True),
                                              (2272, 2864, 1152, True), (4064, 752, 1024, False), (2288, 1520, 640, False), (80, 80, 2048, True)])
def test_256x192_tiles_in_one_round(program, m, n, k, persistent):
    names = subprocess.run(["c++filt"], input="\n".join(program(m, n, k, 1, 0, 0)), check=True, capture_output=True, text=True).stdout
    assert ("tile_gemm_large_kernel<192" in names) == persistent and ("tile_gemm_kernel<256, 192" in names) != persistent, names


# tall groups that are a single round of 256x192 tiles: those, in one launch (of 256x256 tiles, 147 would be too few for one);
# more than a round of them: 256x256
@pytest.mark.parametrize("groups,m,n,k,columns", [(7, 768, 1664, 2176, 192), (4, 512, 4960, 1664, 192), (8, 512, 3584, 2048, 256)])
def test_tall_groups_in_one_round(program, groups, m, n, k, columns):
    names = [name for name in program(m, n, k, 0, groups) if "tile_gemm" in name]
    assert len(names) == 1, names
    name = subprocess.run(["c++filt", names[0]], check=True, capture_output=True, text=True).stdout
    assert f"tile_gemm_large_grouped_kernel<{columns}," in name, name


# small launches of tall groups: a tile per workgroup, with K split where the tiles are few; large ones, narrow N, rows off the
# grid over a hundred K blocks for a CU, a header that is not there: the persistent kernels
@pytest.mark.parametrize("groups,m,n,k,kernel", [(8, 100, 512, 512, "tile_gemm_each_kernel<64, 64, 2, 2, 4, false, true>"),
                                                 (20, 112, 576, 1024, "tile_gemm_each_kernel<64, 64, 2, 2, 4, false, false>"),
                                                 (9, 333, 976, 2048, "tile_gemm_each_kernel<128, 128, 2, 2, 4, false, true>"),
                                                 (8, 1024, 7168, 2048, "tile_gemm_large_grouped_kernel<256"), (8, 100, 240, 512, "tile_gemm_grouped_kernel<"),
                                                 (35, 773, 576, 7168, "tile_gemm_large_grouped_kernel<256")])
def test_tall_groups_with_a_tile_per_workgroup(program, groups, m, n, k, kernel):
    names = subprocess.run(["c++filt"], input="\n".join(program(m, n, k, 0, groups)), check=True, capture_output=True, text=True).stdout
    assert kernel in names, names


def test_a_grouped_call_reports_that_no_workspace_can_be_allocated(program):
    """rows off the grid, K to be split in the process-wide workspace: the runtime's error, before anything is launched"""
    assert program("no-memory", 9, 87, 576, 7168) == ["code", "2"]
