"""Quantisers: the decode batch's kernel (up to 64 rows, every count of rows that its waves and packed block treat in a way of
their own), and the tiles whose k-rows start at any byte.  A row's codes and scales do not depend on the rows beside it: they
are those of the same rows in a taller matrix, which another kernel quantises, and bit for bit the oracle's."""
import numpy as np
import pytest

import oracle
from test_gpu_quantize import _bf16_bits, _say

pytestmark = pytest.mark.gpu


def _quantise(pkg, x, rows, dtype, shift=0):
    import torch
    k = x.shape[1]
    src = np.ascontiguousarray(x[:rows]) if dtype == pkg.DTYPE_F32 else _bf16_bits(x[:rows]).view(np.int16)
    q = torch.full((shift + k * rows + 64,), 0x7F, dtype=torch.uint8, device="cuda")
    s = torch.full((k // 128 * rows + 16,), -1.0, dtype=torch.float32, device="cuda")
    _say(f"[gpu case] quantise rows={rows} k={k} dtype={dtype} q+{shift}")
    pkg.quantize_a_1x128(torch.from_numpy(src).cuda(), q[shift:], s, rows, k, dtype, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (q[:shift] == 0x7F).all() and (q[shift + k * rows:] == 0x7F).all() and (s[k // 128 * rows:] == -1.0).all(), "written outside"
    return q[shift:shift + k * rows].cpu().numpy().reshape(k, rows), s[:k // 128 * rows].cpu().numpy().reshape(k // 128, rows)


@pytest.mark.parametrize("kind", ["bf16", "bf16_f32math", "f32"])
def test_rows_of_a_decode_batch(pkg, kind):
    dtype = {"bf16": pkg.DTYPE_BF16, "bf16_f32math": pkg.DTYPE_BF16_F32MATH, "f32": pkg.DTYPE_F32}[kind]
    k = 640
    x = oracle.gen_normal_bf16(80, k, 4100, 1.0, 50.0)
    x[3, :128] = 0.0
    x[5, 128:256] *= np.float32(2.0 ** -100)
    want_q, want_s = oracle.quantize_a_1x128(x, bf16_arith=kind == "bf16")
    # what the oracle does not define: the tile kernel's codes
    odd = x.copy()
    odd[1, 130], odd[2, 7], odd[9, 300], odd[17, 256:384] = np.inf, -np.inf, np.nan, np.nan
    tall_q, tall_s = _quantise(pkg, odd, 80, dtype)
    for rows in (1, 2, 3, 4, 5, 8, 13, 15, 16, 17, 20, 24, 31, 32, 33, 40, 47, 48, 49, 60, 63, 64):
        q, s = _quantise(pkg, x, rows, dtype)
        assert np.array_equal(s, want_s[:, :rows]) and np.array_equal(q, want_q[:, :rows]), rows
        q, s = _quantise(pkg, odd, rows, dtype)
        assert np.array_equal(s.view(np.uint32), tall_s[:, :rows].view(np.uint32)) and np.array_equal(q, tall_q[:, :rows]), rows


@pytest.mark.parametrize("rows,k,shift", [(1, 128, 4), (24, 256, 8), (63, 256, 1), (65, 256, 0), (79, 384, 0), (100, 256, 3), (127, 128, 0),
                                          (130, 256, 0), (333, 2048, 0), (1023, 7168, 0), (1019, 5120, 5)])
def test_rows_that_start_at_any_byte(pkg, rows, k, shift):
    x = oracle.gen_normal_bf16(rows, k, 4200 + rows, 1.0, 50.0)
    want_q, want_s = oracle.quantize_a_1x128(x, bf16_arith=True)
    q, s = _quantise(pkg, x, rows, pkg.DTYPE_BF16, shift)
    assert np.array_equal(s, want_s) and np.array_equal(q, want_q)
