"""Which calls are refused for want of a workspace: whether a problem runs does not turn on which of two plans level with each
other the estimates prefer.  In a process that sees no device: a call that is not refused ends in the runtime's error."""
import os
import subprocess
import sys

import pytest

CALLS = """
import ctypes as C, sys
L = C.CDLL(sys.argv[1])
devices = C.c_int(0)
L.hipGetDeviceCount(C.byref(devices))
assert devices.value == 0   # the pointers below are made up
vp, i = C.c_void_p, C.c_int
L.fp8_block_gemm_noalloc.argtypes = [vp] * 5 + [i] * 3 + [vp]
L.fp8_block_gemm_ws.argtypes = [vp] * 5 + [i] * 3 + [vp, C.c_size_t, vp]
p, ws = 4096, 1 << 20
for line in sys.stdin:
    entry, m, n, k = line.split()
    m, n, k = int(m), int(n), int(k)
    if entry == "noalloc":
        rc = L.fp8_block_gemm_noalloc(p, p, p, p, p, m, n, k, None)
    else:
        rc = L.fp8_block_gemm_ws(p, p, p, p, p, m, n, k, ws if int(entry) else None, int(entry), None)
    print(rc)
"""

# (bytes of a caller's workspace or the fixed array, m, n, k): unsplit and split plans within a few per cent of each other, with rows on
# and off the grid, on copies (n or m), over strips and tiles
RUN = [("noalloc", 337, 4608, 7168), ("noalloc", 352, 4608, 7168), ("noalloc", 625, 4608, 7168), ("noalloc", 640, 4608, 7168),
       ("noalloc", 833, 1536, 7168), ("noalloc", 1028, 1536, 7168), ("noalloc", 1052, 1536, 7168), ("noalloc", 1889, 1536, 7168),
       ("noalloc", 1619, 576, 7168), ("noalloc", 2722, 576, 7168), ("noalloc", 2805, 576, 7168), ("noalloc", 3154, 512, 7168),
       ("noalloc", 740, 1117, 4864), ("noalloc", 34, 18944, 8320), ("noalloc", 249, 5040, 7040), ("noalloc", 824, 1005, 4736),
       (0, 49, 7168, 2304), (0, 64, 7168, 2304), (0, 306, 688, 3200), (0, 3455, 656, 5120), (0, 1029, 2048, 5888), (0, 625, 4608, 7168),
       (0, 1896, 1536, 7168), (0, 16, 6096, 2432), (0, 28, 10864, 4608), (0, 6006, 96, 3968), (0, 621, 768, 2816), (0, 32, 2880, 4352)]
# a plan without partial sums, or without so many, would take much longer
REFUSED = [(0, 2048, 576, 7168), (0, 1024, 512, 7168), (0, 256, 256, 7168), (16 << 20, 2048, 576, 7168), (0, 33, 100, 128),
           ("noalloc", 8191, 4607, 7168)]


@pytest.fixture(scope="module")
def code(pkg):
    calls = RUN + REFUSED
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")
    done = subprocess.run([sys.executable, "-c", CALLS, pkg.lib_path()], input="".join("%s %d %d %d\n" % c for c in calls), env=env,
                          capture_output=True, text=True, timeout=120, check=True)
    return dict(zip(calls, map(int, done.stdout.split())))


@pytest.mark.parametrize("call", RUN)
def test_a_plan_that_finds_room_runs(code, call):
    assert code[call] > 0, code[call]   # hipErrorNoDevice or the like


@pytest.mark.parametrize("call", REFUSED)
def test_what_needs_a_workspace_says_so(code, call):
    assert code[call] == -4
