"""jitnn_hip_linear_noalloc_dev - the entry point that takes the scratch of a many-row launch from the library's fixed
device array instead of a buffer it may have to allocate - against jitnn_hip_linear_dev on the same inputs: the same
kernels on the same operands, so the same bits.  Calls in a row, each smaller than the first (the array keeps the earlier
calls' contents): the many-row kernel with K slices, the one-pass kernel for 9..64 rows, the GEMV range (no scratch at
all); then the size limit."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import GGML_ID, norm_err, random_valid_blocks

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def jn():
    import jitnn_amd
    jitnn_amd.init()
    return jitnn_amd


def vp(t):
    return C.c_void_p(t.data_ptr())


def run(lib, name, w, x, bias, n):
    y = torch.full((x.shape[0], n), float("nan"), device="cuda")
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = getattr(lib.lib, name)(w.handle, vp(x), x.shape[0], vp(bias) if bias is not None else None, vp(y), st)
    lib.check(rc, name)
    torch.cuda.synchronize()
    return y


def test_noalloc_linear_matches_linear_dev(jn):
    from jitnn_amd import _lib as lib
    assert lib.lib.jitnn_hip_noalloc_scratch_bytes() == 64 << 20
    rng = np.random.default_rng(12)
    g = torch.Generator(device="cuda").manual_seed(12)
    # 4096 x 4096 at 512 rows splits K into slices (partial sums in the scratch); the second call is smaller in every way
    # (then: a ragged Q6_K launch, the one-pass kernel for 9..64 rows of Q4_K / Q5_K / Q4_1 - its prepared operands live in
    # the scratch too -, a 32-value format with rows of odd block counts, and a GEMV call that needs no scratch at all)
    calls = [("Q4_K", 4096, 4096, 512, True), ("Q6_K", 300, 1024, 97, False), ("Q4_K", 640, 2048, 40, True), ("Q5_K", 100, 1024, 17, False),
             ("Q4_1", 250, 1536, 33, True), ("Q8_0", 131, 32 * 9, 70, True), ("Q4_K", 192, 2048, 5, False)]
    for fmt, n, k, rows, with_bias in calls:
        w = jn.Tensor.quantized(jn.DType[fmt], random_valid_blocks(rng, fmt, n, k), n, k)
        x = torch.randn(rows, k, device="cuda", generator=g)
        bias = torch.randn(n, device="cuda", generator=g) if with_bias else None
        ref = run(lib, "jitnn_hip_linear_dev", w, x, bias, n)
        got = run(lib, "jitnn_hip_linear_noalloc_dev", w, x, bias, n)
        assert torch.isfinite(ref).all()
        assert torch.equal(got, ref), (fmt, n, k, rows)
        again = run(lib, "jitnn_hip_linear_noalloc_dev", w, x, bias, n)
        assert torch.equal(again, ref), (fmt, n, k, rows, "second call")


@pytest.mark.parametrize("fmt,n,k,rows", [
    ("Q4_0", 11003, 1056, 513), ("Q4_1", 11005, 1120, 600), ("Q8_0", 12803, 1056, 1025), ("Q5_1", 10930, 1184, 515), ("Q4_K", 11001, 1024, 513),
    ("Q5_K", 11003, 1280, 600), ("Q6_K", 4001, 4096, 1300), ("Q2_K", 11007, 1024, 514), ("Q4_0", 4096, 14336, 2048)])
def test_noalloc_linear_matches_linear_dev_on_dequantised_weights(jn, fmt, n, k, rows):
    """Calls for which jitnn_hip_linear_dev dequantises the weights first (asserted: the thread's scratch holds them) and this entry
    point does not: other kernels, the same FP16 operands and FP32 sums - the same bits, also where the activations of a row
    differ by many orders of magnitude.  Rows, tokens and values per row past whole tiles of every kind."""
    from jitnn_amd import _lib as lib
    rng = np.random.default_rng(n + rows)
    g = torch.Generator(device="cuda").manual_seed(n)
    w = jn.Tensor.quantized(jn.DType[fmt], random_valid_blocks(rng, fmt, n, k), n, k)
    bias = torch.randn(n, device="cuda", generator=g)
    x = torch.randn(rows, k, device="cuda", generator=g) * torch.exp(3 * torch.randn(rows, k, device="cuda", generator=g))
    lib.check(lib.lib.jitnn_hip_thread_release(), "jitnn_hip_thread_release")
    ref = run(lib, "jitnn_hip_linear_dev", w, x, bias, n)
    assert lib.thread_scratch()[0] > 2 * n * k  # (the weights, and the activations beside them)
    got = run(lib, "jitnn_hip_linear_noalloc_dev", w, x, bias, n)
    assert torch.isfinite(ref).all() and torch.equal(got, ref)


def test_noalloc_linear_against_the_oracle_without_allocating_and_under_graph_replay(jn):
    """The entry point against the CPU oracle (not only against its sibling), the property it exists for - a first-ever
    call of a size no earlier call of this process has had leaves the free device memory where it was -, and a many-row
    call captured into a HIP graph: every replay, with eager work between the replays, equals the eager result."""
    from jitnn_amd import _lib as lib
    from oracle import oracle
    rng = np.random.default_rng(14)
    g = torch.Generator(device="cuda").manual_seed(14)
    n, k, rows = 1536, 5120, 600   # (a size no other test of the suite uses)
    raw = random_valid_blocks(rng, "Q4_K", n, k)
    w = jn.Tensor.quantized(jn.DType.Q4_K, raw, n, k)
    x = torch.randn(rows, k, device="cuda", generator=g)
    y = torch.full((rows, n), float("nan"), device="cuda")
    st = torch.cuda.current_stream()
    torch.cuda.synchronize()
    free_before = torch.cuda.mem_get_info()[0]
    lib.check(lib.lib.jitnn_hip_linear_noalloc_dev(w.handle, vp(x), rows, None, vp(y), C.c_void_p(st.cuda_stream)), "noalloc")
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free_before
    sel = np.unique(np.linspace(0, rows - 1, 24).astype(np.int64))
    ref = oracle.gguf_linear(GGML_ID["Q4_K"], x[torch.as_tensor(sel, device="cuda")].cpu().numpy(), raw, None, n, k)
    assert norm_err(y.cpu().numpy()[sel], ref) <= 2e-3   # (more than 64 rows: the FP16 matrix-core path's bar)
    eager = y.clone()
    side = torch.cuda.Stream()
    side.wait_stream(st)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        y.fill_(0)
        with torch.cuda.graph(graph, stream=side):
            lib.check(lib.lib.jitnn_hip_linear_noalloc_dev(w.handle, vp(x), rows, None, vp(y), C.c_void_p(side.cuda_stream)), "noalloc (capture)")
    torch.cuda.synchronize()
    for i in range(3):
        y.fill_(float(i))                      # eager work between the replays
        small = run(lib, "jitnn_hip_linear_noalloc_dev", w, x[:40].contiguous(), None, n)   # the scratch is used by another call in between
        assert torch.isfinite(small).all()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager), i


def test_noalloc_linear_rejects_what_does_not_fit(jn):
    from jitnn_amd import _lib as lib
    rng = np.random.default_rng(13)
    n, k, rows = 64, 16384, 4096  # 4096 x 16384 FP16 activations alone are 128 MiB
    w = jn.Tensor.quantized(jn.DType.Q4_0, random_valid_blocks(rng, "Q4_0", n, k), n, k)
    x = torch.zeros(rows, k, device="cuda")
    y = torch.zeros(rows, n, device="cuda")
    rc = lib.lib.jitnn_hip_linear_noalloc_dev(w.handle, vp(x), rows, None, vp(y), None)
    assert rc == lib.EINVAL and "scratch" in lib.last_error()
    torch.cuda.synchronize()


@pytest.mark.parametrize("fmt,n,k,rows,slices,bias", [
    ("Q4_K", 14336, 4096, 24, 2, True), ("Q6_K", 4096, 14336, 37, 7, False), ("Q6_K", 20000, 2304, 40, 2, True),
    ("Q2_K", 6001, 4352, 33, 3, False), ("Q4_0", 9001, 2816, 25, 2, True), ("Q5_1", 12003, 5888, 40, 3, False), ("Q6_K", 7601, 14336, 5, 7, True)])
def test_captured_linear_without_room_for_its_slices(jn, fmt, n, k, rows, slices, bias):
    """9 to 64 rows (and 5 of long ones) in the kernel that adds up slices of a row, recorded on a thread whose scratch holds the
    operands but not the slices: the same bits as the entry point that allocates nothing and as an eager call.  Short last slices (17
    columns in three, 23 in three, 11 in two), ragged tiles, rows that fill no group of eight."""
    import threading
    from jitnn_amd import _lib as lib
    assert lib.few_rows_slices(GGML_ID[fmt], n, k, rows, adds=bias) == slices
    rng = np.random.default_rng(n)
    w = jn.Tensor.quantized(jn.DType[fmt], random_valid_blocks(rng, fmt, n, k), n, k)
    small = jn.Tensor.quantized(jn.DType[fmt], random_valid_blocks(rng, fmt, 16, k), 16, k)
    g = torch.Generator(device="cuda").manual_seed(k)
    x, b = torch.randn(rows, k, device="cuda", generator=g), torch.randn(n, device="cuda", generator=g) if bias else None
    ref = run(lib, "jitnn_hip_linear_noalloc_dev", w, x, b, n)
    assert torch.isfinite(ref).all() and torch.equal(run(lib, "jitnn_hip_linear_dev", w, x, b, n), ref)
    failed = []

    def work():
        try:
            side = torch.cuda.Stream()
            y, ys = torch.empty_like(ref), torch.empty(rows, 16, device="cuda")

            def call(weight, out, bias):
                lib.check(lib.lib.jitnn_hip_linear_dev(weight.handle, vp(x), rows, vp(bias) if bias is not None else None, vp(out), C.c_void_p(side.cuda_stream)), "linear")

            with torch.cuda.stream(side):
                call(small, ys, None)  # room for the operands of these rows
                side.synchronize()
                held = lib.thread_scratch()[0]
                assert 0 < held < 4 * slices * rows * n
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    call(w, y, b)
                for i in range(3):
                    y.fill_(float("nan"))
                    call(small, ys, None)  # (the scratch is used in between)
                    graph.replay()
                    side.synchronize()
                    assert torch.equal(y, ref), i
                assert lib.thread_scratch() == (held, 0, 1)
                del graph
        except BaseException as e:  # noqa: BLE001 (handed to the test's thread)
            failed.append(e)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    if failed:
        raise failed[0]
