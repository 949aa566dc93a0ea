"""Linears of more than 64 rows at the edges of the kernel that decodes as it goes (prefill.h): one to five steps of K, half a step at the
end of a row, one row past a tile of rows or tokens, both wave layouts (up to 128 rows and beyond) - against FP64 on the oracle's dequantised weights.

Tolerance: weights and activations are rounded to FP16 once each, and the K-quants' scale products once more: at most 3 x 2^-11 of
each product, 1.5e-3 of the sum of their magnitudes, which bounds every output."""
import numpy as np
import pytest
import torch

from helpers import GGML_ID, random_valid_blocks

pytestmark = pytest.mark.gpu


def linear(fmt, n, k, rows, bias, seed=0):
    import jitnn_amd
    from jitnn_amd import _lib as lib
    from oracle import oracle
    jitnn_amd.init()
    rng = np.random.default_rng([seed, n, k, rows])
    raw = random_valid_blocks(rng, fmt, n, k)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32) if bias else None
    w = jitnn_amd.Tensor.quantized(jitnn_amd.DType[fmt], raw, n, k)
    xd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda() if bias else None
    out = []
    for name in ("jitnn_hip_linear_dev", "jitnn_hip_linear_noalloc_dev"):
        y = torch.full((rows * n + 4,), float("nan"), device="cuda")
        lib.check(getattr(lib.lib, name)(w.handle, xd.data_ptr(), rows, bd.data_ptr() if bias else None, y.data_ptr(), None), name)
        torch.cuda.synchronize()
        assert torch.isnan(y[rows * n:]).all()
        out.append(y[:rows * n].reshape(rows, n).cpu().numpy())
    wd = oracle.dequantize(GGML_ID[fmt], raw, n * k).reshape(n, k).astype(np.float64)
    x64 = x.astype(np.float64)
    ref = x64 @ wd.T + (b.astype(np.float64) if bias else 0.0)
    bound = 1.5e-3 * (np.abs(x64) @ np.abs(wd).T) + 1e-6 * np.abs(ref).max()
    assert (np.abs(out[0] - ref) <= bound).all()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("rows", [65, 129, 257])
@pytest.mark.parametrize("fmt,k", [("Q4_0", 32), ("Q4_0", 96), ("Q4_1", 64), ("Q4_1", 160), ("Q8_0", 128), ("Q8_0", 224), ("Q8_0", 320), ("Q5_1", 96),
                                   ("Q4_K", 256), ("Q5_K", 256), ("Q5_K", 512), ("Q6_K", 256), ("Q6_K", 768)])
def test_short_rows_of_k(fmt, k, rows):
    linear(fmt, 132, k, rows, False)


@pytest.mark.parametrize("fmt,n,k,rows,bias", [("Q4_1", 1249, 1120, 130, True), ("Q4_0", 259, 5632, 515, False), ("Q8_0", 1030, 2720, 70, True), ("Q8_0", 1, 8192, 66, False),
                                               ("Q4_K", 1027, 3328, 129, False), ("Q6_K", 301, 6912, 65, True), ("Q5_K", 2002, 4352, 257, False), ("Q6_K", 3328, 2304, 200, True),
                                               ("Q5_1", 515, 3104, 100, False), ("Q2_K", 515, 3072, 100, True)])
def test_slices_of_k(fmt, n, k, rows, bias):
    """Launches cut into slices of K, a last slice shorter than the others among them, with outputs of any length (their slices are joined
    value by value), a bias in the join."""
    linear(fmt, n, k, rows, bias, 1)


def test_captured_without_room_for_the_slices():
    """Recorded on a thread whose scratch holds the activations' operands but not the slices of K, a launch of one weight takes fewer
    slices: the same sums in another order.  FP32 sums of 4096 products, 2^-24 each: 1e-5 of the largest output."""
    import ctypes as C
    import threading
    import jitnn_amd
    from jitnn_amd import _lib as lib
    jitnn_amd.init()
    rows, n, k = 130, 2101, 4096
    rng = np.random.default_rng(3)
    w, small = (jitnn_amd.Tensor.quantized(jitnn_amd.DType.Q8_0, random_valid_blocks(rng, "Q8_0", m, k), m, k) for m in (n, 32))
    x = torch.randn(rows, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    eager, y = torch.empty(rows, n, device="cuda"), torch.empty(rows, n, device="cuda")

    def call(weight, out, stream):
        lib.check(lib.lib.jitnn_hip_linear_dev(weight.handle, C.c_void_p(x.data_ptr()), rows, None, C.c_void_p(out.data_ptr()), C.c_void_p(stream.cuda_stream)), "linear")

    call(w, eager, torch.cuda.current_stream())
    torch.cuda.synchronize()
    failed = []

    def work():
        try:
            side = torch.cuda.Stream()
            with torch.cuda.stream(side):
                call(small, torch.empty(rows, 32, device="cuda"), side)
                side.synchronize()
                held = lib.thread_scratch()[0]
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    call(w, y, side)
                for i in range(3):
                    y.fill_(float("nan"))
                    graph.replay()
                    side.synchronize()
                    assert (y - eager).abs().max() <= 1e-5 * eager.abs().max(), i
                assert lib.thread_scratch()[0] == held
                del graph
        except BaseException as e:  # noqa: BLE001 (handed to the test's thread)
            failed.append(e)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    if failed:
        raise failed[0]
