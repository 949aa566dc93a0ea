"""Linears of a few activation rows on rows of 32-value blocks that are not whole 256-value columns: the whole columns in the one-pass kernels,
the last one to seven blocks in gemv_tail_kernel - one column and many, ragged last tiles of weight rows, both ends of the range of activation
rows, bias, one slice of K and several - against FP64 on the oracle's dequantised weights; and recorded on a thread without scratch.

Tolerance: as in test_gpu_rows_held.py - two FP16 parts of a row (2^-22 per product) and about log2(K) roundings of 2^-24 of its FP32 sums - 2e-6 of
the largest output for K up to 13000."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

from helpers import GGML_ID, norm_err, random_valid_blocks

pytestmark = pytest.mark.gpu


def call(lib, name, w, x, b, y, stream=None):
    lib.check(getattr(lib.lib, name)(w.handle, x.data_ptr(), x.shape[0], b.data_ptr() if b is not None else None, y.data_ptr(),
                                     C.c_void_p(stream.cuda_stream) if stream else None), name)


@pytest.mark.parametrize("fmt,n,k,rows,bias", [
    ("Q8_0", 16, 288, 9, False), ("Q4_0", 17, 480, 64, True), ("Q4_1", 300, 1056, 13, False), ("Q8_0", 1001, 2016, 33, True), ("Q4_0", 2050, 2272, 9, False),
    ("Q4_1", 515, 3296, 5, True), ("Q8_0", 130, 7008, 8, False), ("Q4_0", 4099, 4064, 41, False), ("Q4_1", 96, 12704, 3, True), ("Q8_0", 260, 12960, 64, True)])
def test_ragged_rows_match_the_oracle(fmt, n, k, rows, bias):
    import jitnn_amd
    from jitnn_amd import _lib as lib
    from oracle import oracle
    jitnn_amd.init()
    rng = np.random.default_rng([n, k, rows])
    raw = random_valid_blocks(rng, fmt, n, k)
    x = rng.standard_normal((rows, k)).astype(np.float32) * np.exp(2 * rng.standard_normal((rows, 1))).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32) if bias else None
    w = jitnn_amd.Tensor.quantized(jitnn_amd.DType[fmt], raw, n, k)
    xd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda() if bias else None
    out = []
    for name in ("jitnn_hip_linear_dev", "jitnn_hip_linear_noalloc_dev"):
        y = torch.full((rows, n), float("nan"), device="cuda")
        call(lib, name, w, xd, bd, y)
        torch.cuda.synchronize()
        out.append(y.cpu().numpy())
    ref = x.astype(np.float64) @ oracle.dequantize(GGML_ID[fmt], raw, n * k).reshape(n, k).astype(np.float64).T + (b.astype(np.float64) if bias else 0.0)
    for r in range(rows):
        assert norm_err(out[0][r], ref[r]) <= 2e-6, r
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("fmt", ["Q4_0", "Q4_1", "Q8_0"])
@pytest.mark.parametrize("k,rows,few", [(480, 24, 8), (1056, 16, 8), (2272, 40, 8), (5088, 24, 4), (11456, 40, 4), (14304, 10, 2)])
def test_no_further_off_than_in_passes(fmt, k, rows, few):
    """The same rows a few at a time take the kernels that multiply in FP32: in one pass the call is at most as far from FP64 (2-norm over 40000
    outputs and more), on weights around zero, where the offsets of Q4_1 and the sums of its quants all but cancel."""
    import jitnn_amd
    from jitnn_amd import _lib as lib
    from oracle import oracle
    jitnn_amd.init()
    n = 4000
    rng = np.random.default_rng([k, rows])
    raw = random_valid_blocks(rng, fmt, n, k)
    if fmt == "Q4_1":
        blocks = raw.reshape(-1, 20)
        blocks[:, 2:4] = (-7.5 * blocks[:, :2].copy().view(np.float16).astype(np.float32)).astype(np.float16).view(np.uint8)
    w = jitnn_amd.Tensor.quantized(jitnn_amd.DType[fmt], raw, n, k)
    x = torch.randn(rows, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(k))
    whole, parts = torch.empty(rows, n, device="cuda"), torch.empty(rows, n, device="cuda")
    call(lib, "jitnn_hip_linear_dev", w, x, None, whole)
    for r in range(0, rows, few):
        call(lib, "jitnn_hip_linear_dev", w, x[r:r + few], None, parts[r:r + few])
    torch.cuda.synchronize()
    ref = x.double() @ torch.from_numpy(oracle.dequantize(GGML_ID[fmt], raw, n * k).reshape(n, k)).cuda().double().T
    assert (whole - ref).norm() <= (parts - ref).norm()


def test_captured_without_scratch():
    """A thread whose first call is recorded has no scratch: the passes of eight rows, the same products in FP32-grade arithmetic of another kind."""
    import jitnn_amd
    from jitnn_amd import _lib as lib
    jitnn_amd.init()
    n, k, rows = 520, 1120, 21
    w = jitnn_amd.Tensor.quantized(jitnn_amd.DType.Q4_1, random_valid_blocks(np.random.default_rng(5), "Q4_1", n, k), n, k)
    x = torch.randn(rows, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(5))
    eager, y = torch.empty(rows, n, device="cuda"), torch.empty(rows, n, device="cuda")
    call(lib, "jitnn_hip_linear_dev", w, x, None, eager)
    torch.cuda.synchronize()
    failed = []

    def work():
        try:
            side = torch.cuda.Stream()
            with torch.cuda.stream(side):
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    call(lib, "jitnn_hip_linear_dev", w, x, None, y, side)
                for i in range(3):
                    y.fill_(float("nan"))
                    graph.replay()
                    side.synchronize()
                    assert (y - eager).abs().max() <= 4e-6 * eager.abs().max(), i
                assert lib.thread_scratch()[0] == 0
                del graph
        except BaseException as e:  # noqa: BLE001 (handed to the test's thread)
            failed.append(e)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    if failed:
        raise failed[0]
