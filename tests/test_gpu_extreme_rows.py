"""Activation rows at both ends of the FP32 range, subnormal ones and one whose largest value is near the largest number, through every kernel that scales a row or a column of it by a power
of two before it goes to FP16: the scale itself has to stay a finite number.  Each row against FP64 on the oracle's dequantised
weights; the other rows of the call are ordinary.

Tolerance: that of the kernel at ordinary magnitudes - 2e-6 of the row's largest output up to 64 rows, 1.5e-3 of the sum of the products'
magnitudes beyond (FP16 operands) - and, where outputs are subnormal, 2^-150 for each of the up to 100 FP32 sums on the way, and what FP16's smallest
step, 2^-24, is worth in a block's sum of x (scaled by 2^126 / 64, rounded by half of it: 2^-145) times the offset it meets, the value of
a quant of zero: at most K / 16 times the largest weight."""
import numpy as np
import pytest
import torch

from helpers import GGML_ID, random_valid_blocks

pytestmark = pytest.mark.gpu

SIZES = (1e-30, 1e-36, 1e-40, 3e-44)


@pytest.mark.parametrize("fmt,n,k,rows", [
    ("Q8_0", 300, 1056, 9), ("Q4_0", 130, 2272, 33), ("Q4_1", 96, 3296, 64),  # rows that are no whole columns: rows_prepare_kernel and the tail
    ("Q4_K", 83, 2304, 7), ("Q8_0", 83, 2304, 8),  # gemv_mfma_kernel
    ("Q4_K", 300, 4096, 40), ("Q6_K", 515, 2304, 48), ("Q4_1", 64, 1024, 12),  # rows_prepare_kernel, both kernels behind it
    ("Q4_K", 300, 4096, 70), ("Q8_0", 64, 16672, 100)])  # x_prepare_kernel; longer rows: x_row_scale_kernel and x_to_operand_kernel
def test_rows_at_the_ends_of_the_range(fmt, n, k, rows):
    import jitnn_amd
    from jitnn_amd import _lib as lib
    from oracle import oracle
    jitnn_amd.init()
    rng = np.random.default_rng([n, k, rows])
    raw = random_valid_blocks(rng, fmt, n, k, lo=2e-5, hi=1e-4)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    for r, size in enumerate(SIZES):
        x[r] = (x[r].astype(np.float64) * size).astype(np.float32)
    x[4] *= np.float32(1e34)
    x[4, 200] = np.float32(3.3e38)
    w = jitnn_amd.Tensor.quantized(jitnn_amd.DType[fmt], raw, n, k)
    xd, y = torch.from_numpy(x).cuda(), torch.full((rows, n), float("nan"), device="cuda")
    lib.check(lib.lib.jitnn_hip_linear_dev(w.handle, xd.data_ptr(), rows, None, y.data_ptr(), None), "linear")
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    wd, x64 = oracle.dequantize(GGML_ID[fmt], raw, n * k).reshape(n, k).astype(np.float64), x.astype(np.float64)
    ref = x64 @ wd.T
    for r in range(rows):
        bound = 2e-6 * np.abs(ref[r]).max() if rows <= 64 else 1.5e-3 * (np.abs(x64[r]) @ np.abs(wd).T)
        assert (np.abs(got[r] - ref[r]) <= bound + 100 * 2.0**-150 + k / 16 * 2.0**-145 * np.abs(wd).max()).all(), (r, float(np.abs(x[r]).max()))
