"""K splits added inside the tile kernels with four multiplying waves, whose copy waves gather half of the patches: every
number of senders around a trip, cut tiles, rows off the grid, bit for bit what the reduction kernel adds, launch after launch."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import _assert_every_element, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant,ksplit,m,n,k", [
    *((4, s, 80, 144, 128 * (2 * s - 1)) for s in (2, 3, 4, 5, 6, 7, 8)),   # the last split a block short
    (4, 4, 64, 64, 512), (4, 3, 77, 208, 1024), (4, 8, 117, 80, 2048),              # one block each; rows off the grid
    (2, 2, 333, 2816, 3072), (2, 3, 269, 2048, 4736), (2, 5, 141, 1664, 7680), (2, 2, 145, 384, 7168),  # rows off the grid
    (2, 2, 144, 256, 2048), (2, 2, 144, 256, 1792), (2, 2, 333, 256, 2816),          # either side of where four waves take over
    (2, 2, 144, 208, 4096), (2, 3, 256, 144, 6016), (2, 4, 128, 128, 8192), (2, 2, 400, 272, 3968)])
def test_splits_added_by_eight_waves(pkg, variant, ksplit, m, n, k):
    kernel = 0 if m % 16 else pkg.KERNEL_SPLITK   # by name no rows off the grid
    a, b, sa, sb = oracle.make_inputs(m, n, k, 3100 + m + n + k, 0.5, 30.0)
    want, name = _run(pkg, a, b, sa, sb, m, n, k, kernel=kernel, variant=variant, ksplit=ksplit, fused=0)
    _assert_every_element(want, a, b, sa, sb, m, n, k, name)
    for _ in range(3):   # what a launch left in the mailbox, the next one would take for its own
        got, fused = _run(pkg, a, b, sa, sb, m, n, k, kernel=kernel, variant=variant, ksplit=ksplit, fused=1)
        assert fused == name + "f", fused
        assert np.array_equal(want, got), f"{fused}: differs from the reduction kernel's result"
