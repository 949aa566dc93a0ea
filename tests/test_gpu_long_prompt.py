"""The routes of long prompts - weights dequantised first, then a plain FP16 product - at the sizes where their tiles can go
wrong, against the oracle's dequantised values in FP64 and against the same prompt in short passes."""
import numpy as np
import pytest

from helpers import GGML_ID, norm_err, random_valid_blocks
from test_gpu_decode import MIX, build

pytestmark = pytest.mark.gpu

MFMA_BAR = 2e-3  # FP16 operands, FP32 accumulation: the bar of the many-row path


@pytest.fixture(scope="module")
def jn():
    import jitnn_amd
    jitnn_amd.init()
    return jitnn_amd


# ragged rows, tokens and K steps (32 past a whole 64), row counts that are no multiple of four; the last column: weight rows
# per tile of the kernel on dequantised weights
CASES = [("Q4_0", 11003, 1056, 513, 192), ("Q4_1", 11005, 1120, 600, 192), ("Q8_0", 11004, 1024, 768, 192), ("Q5_1", 10930, 1184, 515, 192),
         ("Q4_K", 11001, 1024, 513, 192), ("Q5_K", 11003, 1280, 600, 192), ("Q6_K", 11136, 1024, 701, 192), ("Q2_K", 11007, 1024, 514, 192),
         ("Q8_0", 2101, 4096, 3900, 192), ("Q8_0", 12803, 1056, 1025, 256), ("Q8_0", 2751, 1056, 1300, 128), ("Q6_K", 4001, 4096, 1300, 128)]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("fmt,n,k,rows,tile", CASES)
def test_linear_many_rows(jn, fmt, n, k, rows, tile, bias):
    from jitnn_amd import _lib as lib
    from oracle import oracle
    assert lib.many_row_tile([(GGML_ID[fmt], n)], k, rows) == tile
    rng = np.random.default_rng(n + k + rows)
    raw = random_valid_blocks(rng, fmt, n, k)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[0] *= 1e4
    x[1] *= 1e-6
    b = rng.standard_normal(n).astype(np.float32) if bias else None
    y = jn.Gguf.linear(jn.Tensor.of(x), jn.Tensor.quantized(jn.DType[fmt], raw, n, k), jn.Tensor.of(b) if bias else None).numpy()
    w = oracle.dequantize(GGML_ID[fmt], raw, n * k).reshape(n, k).astype(np.float64)
    ref = x.astype(np.float64) @ w.T
    wnorm = float(np.sqrt((w ** 2).sum() / n))
    got = y.astype(np.float64) - (b if bias else 0.0)
    for r in range(rows):  # row by row, against the larger of its biggest output and |x_r| * rms row norm of W
        scale = max(float(np.abs(ref[r]).max()), float(np.linalg.norm(x[r].astype(np.float64))) * wnorm, 1e-30)
        assert np.abs(got[r] - ref[r]).max() <= MFMA_BAR * scale + (1e-6 * np.abs(b).max() if bias else 0.0), (fmt, r)


def test_long_prompt_equals_short_passes(jn):
    """2900 tokens through one layer, whose q, k | v and gate | up launches take the dequantised route (attn_o and down do not:
    too few tiles; test_whole_layer_on_dequantised_weights has them), against the same tokens in passes of 256, where none does.  Both round the same operands to FP16 and add up in FP32, in another order;
    what differs before one rounding (2^-11) differs by one after it: the bar of one linear."""
    cfg = dict(layers=1, d_model=1024, heads=32, kv_heads=8, head_dim=64, ffn=1536, vocab=512, max_ctx=2900, rms_eps=1e-5, rope_theta=1e4)
    dec, *_ = build(jn, cfg, 4)
    x = np.random.default_rng(6).standard_normal((2900, cfg["d_model"])).astype(np.float32)
    whole = dec.prefill(x, 0)
    k1, v1 = dec.kv_read(0, 0, 2900)
    for p in range(0, 2900, 256):
        parts = dec.prefill(x[p:p + 256], p)
    k2, v2 = dec.kv_read(0, 0, 2900)
    for a, b in ((k1, k2), (v1, v2), (whole, parts)):
        assert np.isfinite(a).all() and norm_err(a, b) <= MFMA_BAR, norm_err(a, b)
    dec.close()


def test_capture_without_room_for_the_dequantised_weights(jn):
    """Scratch that fits the operands of the kernel that decodes as it goes, but not dequantised weights beside them, cannot
    grow under a stream capture: the launch takes the former kernel.  In a thread of its own, whose scratch starts empty."""
    import ctypes as C
    import threading
    import torch
    from jitnn_amd import _lib as lib

    rows, n, k = 3900, 2101, 4096  # (the Q8_0 case above: dequantised first when called eagerly)
    rng = np.random.default_rng(8)
    small = jn.Tensor.quantized(jn.DType.Q8_0, random_valid_blocks(rng, "Q8_0", 32, k), 32, k)
    w = jn.Tensor.quantized(jn.DType.Q8_0, random_valid_blocks(rng, "Q8_0", n, k), n, k)
    x = torch.randn(rows, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(8))
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
                call(small, torch.empty(rows, 32, device="cuda"), side)  # the activations' operands: 32 MiB of scratch
                side.synchronize()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    call(w, y, side)
                for i in range(3):
                    y.fill_(float("nan"))
                    graph.replay()
                    side.synchronize()
                    assert torch.equal(y, eager), i  # the same FP16 operands, the same FP32 sums
                del graph
        except BaseException as e:  # noqa: BLE001 (handed to the test's thread)
            failed.append(e)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    if failed:
        raise failed[0]


def in_thread(work):
    """Runs work() in a thread of its own, whose scratch starts empty, and raises here what it raises there."""
    import threading
    failed = []

    def body():
        try:
            work()
        except BaseException as e:  # noqa: BLE001 (handed to the test's thread)
            failed.append(e)

    t = threading.Thread(target=body)
    t.start()
    t.join()
    if failed:
        raise failed[0]


@pytest.mark.parametrize("case", ["same_call", "wider_weight", "more_rows"])
def test_recorded_linear_outlives_scratch_growth(jn, case):
    """A long linear recorded into a graph, then an eager call on the same thread that needs more scratch: the same call, which
    only now finds room for dequantised weights; a weight of more rows; more activations.  The recorded block is kept, so a
    replay after each gives the eager bits."""
    import ctypes as C
    import torch
    from jitnn_amd import _lib as lib

    rng = np.random.default_rng(9)
    k = 4096
    raw = {n: random_valid_blocks(rng, "Q8_0", n, k) for n in (32, 2101, 4200)}
    w = {n: jn.Tensor.quantized(jn.DType.Q8_0, r, n, k) for n, r in raw.items()}
    gen = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn(3900, k, device="cuda", generator=gen)
    longer = torch.randn(4700, k, device="cuda", generator=gen)

    def call(n, xs, out, stream):
        lib.check(lib.lib.jitnn_hip_linear_dev(w[n].handle, C.c_void_p(xs.data_ptr()), xs.shape[0], None, C.c_void_p(out.data_ptr()), C.c_void_p(stream.cuda_stream)), "linear")

    ref = torch.empty(3900, 2101, device="cuda")
    call(2101, x, ref, torch.cuda.current_stream())
    torch.cuda.synchronize()

    def work():
        side = torch.cuda.Stream()
        y = torch.empty_like(ref)
        with torch.cuda.stream(side):
            call(32 if case == "same_call" else 2101, x, torch.empty(3900, 4200, device="cuda"), side)
            side.synchronize()
            assert lib.thread_scratch()[1] == 0
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                call(2101, x, y, side)
            for i in range(3):
                if case == "same_call":
                    again = torch.empty_like(ref)
                    call(2101, x, again, side)
                elif case == "wider_weight":
                    call(4200, x, torch.empty(3900, 4200, device="cuda"), side)
                else:
                    call(2101, longer, torch.empty(4700, 2101, device="cuda"), side)
                side.synchronize()
                held, kept, _ = lib.thread_scratch()
                # (the same call needs more of the other block only: nothing recorded is outgrown)
                assert (kept == 0) if case == "same_call" else (0 < kept < held), (held, kept)
                y.fill_(float("nan"))
                graph.replay()
                side.synchronize()
                assert torch.equal(y, ref), i
                if case == "same_call":
                    assert torch.equal(again, ref), i
            del graph

    in_thread(work)


LONG = dict(layers=1, d_model=1280, heads=16, kv_heads=2, head_dim=128, ffn=1792, vocab=512, max_ctx=3100, rms_eps=1e-5, rope_theta=1e4)
TWO_FORMATS = {**MIX, "ffn_up": "Q5_K"}  # gate and up in one launch, but not as one product


@pytest.mark.parametrize("mix", [MIX, TWO_FORMATS], ids=["one_product", "two_formats"])
def test_prompt_pass_grows_the_scratch_once(jn, mix):
    """The largest launch of the layer is gate and up: the scratch is sized for it before the first launch, also where the two
    have formats of their own.  One allocation for the operands, one for the weights."""
    from jitnn_amd import _lib as lib
    dec, *_ = build(jn, LONG, 4, mix)
    x = np.random.default_rng(6).standard_normal((3100, LONG["d_model"])).astype(np.float32)

    def work():
        dec.prefill(x, 0)
        assert lib.thread_scratch()[2] == 2, lib.thread_scratch()

    in_thread(work)
    dec.close()


# rows of every weight, and values per row, 32 past a multiple of 128: whole and ragged tiles of every launch, K steps past the end
RAGGED = {**LONG, "d_model": 1184, "ffn": 1312}


@pytest.mark.parametrize("cfg,mix,tiles", [(LONG, MIX, (192, 128, 256, 128)), (LONG, TWO_FORMATS, (192, 128, 256, 128)),
                                           (RAGGED, dict.fromkeys(MIX, "Q8_0"), (192, 128, 256, 128))], ids=["one_product", "two_formats", "ragged"])
def test_whole_layer_on_dequantised_weights(jn, cfg, mix, tiles):
    """3100 tokens (28 past whole tiles) through two layers whose four launches all take the dequantised route: q, k and v; attn_o
    with the residual; gate and up as one product with the SwiGLU, or as two weights whose SwiGLU is formed by the preparation
    of down's activations; down with the residual.  Against the same tokens in passes of 256, where none of them does:
    the same FP16 operands and FP32 sums, in another order where the short passes split K, attention in other chunks, and the last
    28 tokens on FP32-grade kernels - the bar of one linear.  The second layer's keys and values are made of every token's output of the first: whole and ragged tiles."""
    from jitnn_amd import _lib as lib
    d, qd, kd, ffn, T = cfg["d_model"], cfg["heads"] * cfg["head_dim"], cfg["kv_heads"] * cfg["head_dim"], cfg["ffn"], 3100
    one = mix["ffn_gate"] == mix["ffn_up"]
    f = {slot: GGML_ID[name] for slot, name in mix.items()}

    def routes(tokens):
        return (lib.many_row_tile([(f["attn_q"], qd), (f["attn_k"], kd), (f["attn_v"], kd)], d, tokens), lib.many_row_tile([(f["attn_o"], d)], qd, tokens, residual=True),
                lib.many_row_tile([(f["ffn_gate"], ffn), (f["ffn_up"], ffn)], d, tokens, gate_up=one), lib.many_row_tile([(f["ffn_down"], d)], ffn, tokens, residual=True))

    assert routes(T) == tiles and routes(256) == (0, 0, 0, 0)
    dec, *_ = build(jn, {**cfg, "layers": 2}, 4, mix, "Q8_0")
    x = np.random.default_rng(6).standard_normal((T, d)).astype(np.float32)
    got = {}

    def whole():
        got["logits"] = dec.prefill(x, 0)
        assert lib.thread_scratch()[2] == 2  # (one block for the operands, one for the weights: the route was not refused)

    in_thread(whole)
    kv = [*dec.kv_read(0, 0, T), *dec.kv_read(1, 0, T)]
    for p in range(0, T, 256):
        parts = dec.prefill(x[p:p + 256], p)
    for a, b in zip(kv + [got["logits"]], [*dec.kv_read(0, 0, T), *dec.kv_read(1, 0, T), parts]):
        assert np.isfinite(a).all() and norm_err(a, b) <= MFMA_BAR, norm_err(a, b)
    dec.close()
