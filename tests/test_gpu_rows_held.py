"""Linears of 9..64 rows (3 of long ones) at the edges of the kernel that holds the activation operands in registers (gemv_held.h): rows of one
256-value column (every wave a tile of its own), of numbers of columns that leave waves or the last slice short, ragged last
tiles, more steps than one per workgroup, groups of rows shared out unevenly, the join of several slices and of one with a bias -
against FP64 on the oracle's dequantised weights.  The route of every launch is asserted (the number of slices of a row).

Tolerance: a row's operands carry 22 bits (two FP16 parts), the sums of a column are FP32 and the columns' meet in FP32:
2^-22 per product and about log2(K) roundings of 2^-24 on the way, against the largest output - 2e-6 for K up to 11008."""
import numpy as np
import pytest
import torch

from helpers import GGML_ID, norm_err, random_valid_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,n,k,rows,bias,slices", [
    ("Q6_K", 16, 256, 9, False, 1), ("Q6_K", 4111, 256, 33, False, 1), ("Q6_K", 300, 512, 64, False, 1), ("Q6_K", 1000, 768, 40, False, 1),
    ("Q6_K", 2001, 1280, 17, True, 1), ("Q6_K", 4500, 2048, 41, False, 1), ("Q6_K", 515, 2304, 48, False, 2), ("Q6_K", 130, 11008, 37, True, 6),
    ("Q6_K", 96, 14336, 3, False, 7), ("Q4_K", 6001, 1536, 40, False, 1), ("Q5_K", 5003, 2816, 57, True, 2), ("Q2_K", 6002, 1536, 23, False, 1),
    ("Q4_0", 24003, 2048, 25, False, 1), ("Q4_1", 24001, 2048, 12, False, 1), ("Q8_0", 24005, 2048, 39, False, 1), ("Q8_0", 4500, 512, 40, True, 1),
    ("Q5_1", 12009, 5888, 40, True, 3), ("Q5_1", 12009, 1792, 40, False, 1)])
def test_held_rows_match_the_oracle(fmt, n, k, rows, bias, slices):
    import jitnn_amd
    from jitnn_amd import _lib as lib
    from oracle import oracle
    jitnn_amd.init()
    assert lib.few_rows_slices(GGML_ID[fmt], n, k, rows, adds=bias) == slices
    rng = np.random.default_rng(n + rows)
    raw = random_valid_blocks(rng, fmt, n, k)
    x = rng.standard_normal((rows, k)).astype(np.float32) * np.exp(2 * rng.standard_normal((rows, 1))).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32) if bias else None
    w = jitnn_amd.Tensor.quantized(jitnn_amd.DType[fmt], raw, n, k)
    xd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda() if bias else None
    out = []
    for name in ("jitnn_hip_linear_dev", "jitnn_hip_linear_noalloc_dev", "jitnn_hip_linear_dev"):
        y = torch.full((rows, n), float("nan"), device="cuda")
        rc = getattr(lib.lib, name)(w.handle, xd.data_ptr(), rows, bd.data_ptr() if bias else None, y.data_ptr(), None)
        lib.check(rc, name)
        torch.cuda.synchronize()
        out.append(y.cpu().numpy())
    wd = oracle.dequantize(GGML_ID[fmt], raw, n * k).reshape(n, k).astype(np.float64)
    ref = x.astype(np.float64) @ wd.T + (b.astype(np.float64) if bias else 0.0)
    assert np.isfinite(out[0]).all()
    for r in range(rows):  # row by row: their magnitudes differ
        assert norm_err(out[0][r], ref[r]) <= 2e-6, r
    assert np.array_equal(out[1], out[0]) and np.array_equal(out[2], out[0])
