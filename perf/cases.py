"""The work a user of jitnn_amd has it do, as cases that can be timed: linears on quantised weights at one row (a decode
step), a few rows (a batch) and many rows (a prompt), a whole model's decode step and prompt pass, the dequantiser and the
Q8_0 quantiser, and a linear on host tensors.  The entry points are the package's: the device-pointer functions of its C
library (through jitnn_amd._lib, as bench.py calls them), LlamaDecoder, and Gguf.linear on host tensors.

Weights are blocks whose dequantised values are about N(0, 0.02), activations N(0, 1), keys and values N(0, 1).
"""
import ctypes as C
import math
import weakref

import torch

import jitnn_amd
from jitnn_amd import _lib

BLOCK = {"Q8_0": (8, 32, 34), "Q4_0": (2, 32, 18), "Q4_1": (3, 32, 20), "Q4_K": (12, 256, 144), "Q5_K": (13, 256, 176), "Q6_K": (14, 256, 210)}

# which format the seven projections of a layer (q, k, v, o, gate, up, down) and the output head have in a file of that mix
MIX = {"Q4_K_M": ("Q4_K", "Q4_K", "Q6_K", "Q4_K", "Q4_K", "Q4_K", "Q6_K", "Q6_K"),
       "Q5_K_M": ("Q5_K", "Q5_K", "Q6_K", "Q5_K", "Q5_K", "Q5_K", "Q6_K", "Q6_K"),
       "Q8_0": ("Q8_0",) * 8,
       "Q4_0": ("Q4_0",) * 7 + ("Q6_K",)}

# 32 layers, d_model 4096, 32 query heads over 8 key / value heads of 128, FFN 14336, vocabulary 128256: the Llama-8B shape
SHAPE_8B = dict(layers=32, d=4096, heads=32, kv=8, hd=128, ffn=14336, vocab=128256, mix="Q4_K_M")


def nbytes(fmt, n, k):
    _, qk, nb = BLOCK[fmt]
    return n * (k // qk) * nb


def listed():
    return [
        # the smallest call: one token through a square Q8_0 projection, one call per layer
        dict(name="linear_q8_0_4096x4096_r1", kind="linear", fmt="Q8_0", n=4096, k=4096, rows=1, bias=False, stack=8),
        # one token through the FFN up-projections of an 8B model: the largest weight of a decode step
        dict(name="linear_q4_k_14336x4096_r1", kind="linear", fmt="Q4_K", n=14336, k=4096, rows=1, bias=False, stack=8),
        # four sequences decoded together, a 7B model's FFN up-projection, with a bias
        dict(name="linear_q4_0_11008x4096_r4", kind="linear", fmt="Q4_0", n=11008, k=4096, rows=4, bias=True, stack=8),
        # eight sequences decoded together
        dict(name="linear_q4_k_14336x4096_r8", kind="linear", fmt="Q4_K", n=14336, k=4096, rows=8, bias=False, stack=8),
        # a short prompt or a larger batch through the FFN down-projections: a ragged number of rows
        dict(name="linear_q6_k_4096x14336_r37", kind="linear", fmt="Q6_K", n=4096, k=14336, rows=37, bias=False, stack=4),
        # a caller with host tensors: x goes up and y comes back on every call (Gguf.linear)
        dict(name="host_linear_q4_k_14336x4096_r1", kind="host", fmt="Q4_K", n=14336, k=4096, rows=1, bias=False),
        # one greedy token of the 8B model (embedding row, all layers over the cache, arg-max), 512 tokens into a context
        dict(name="decode_8b_ctx512", kind="decode", ctx=512, interleaved=False, **SHAPE_8B),
        # the same deep into a long context
        dict(name="decode_8b_ctx4000", kind="decode", ctx=4000, interleaved=False, **SHAPE_8B),
        # a prompt of one sentence
        dict(name="prefill_8b_40", kind="prefill", tokens=40, pos0=0, interleaved=False, **SHAPE_8B),
        # a prompt of a page
        dict(name="prefill_8b_512", kind="prefill", tokens=512, pos0=0, interleaved=False, **SHAPE_8B),
        # a prompt that fills the default context
        dict(name="prefill_8b_4096", kind="prefill", tokens=4096, pos0=0, interleaved=False, **SHAPE_8B),
        # a weight converted: dequantised to FP32 and quantised to Q8_0
        dict(name="requantize_q4_k_14336x4096", kind="codec", fmt="Q4_K", n=14336, k=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _row_length(rng, fmt, lo, hi):
    """A row of whole 256-value blocks, or - where the blocks hold 32 values - of any number of those."""
    qk = 256 if BLOCK[fmt][1] == 256 or rng.random() < 0.7 else 32
    return max(1, _log(rng, lo, hi) // qk) * qk


def draw(rng):
    kind = rng.choices(("linear", "host", "codec", "decode", "prefill"), (10, 1, 2, 3, 4))[0]
    if kind in ("linear", "host", "codec"):
        fmt = rng.choice(sorted(BLOCK))
        k = _row_length(rng, fmt, 1024, 14336)
        n = min(_log(rng, 512, 32768), 14336 * 4096 // k)
        n = n if rng.random() < 0.4 else max(256, n // 256 * 256)
        if kind == "codec":
            return dict(kind=kind, fmt=fmt, n=n, k=k)
        rows = rng.choice((1, rng.randint(2, 8), rng.randint(9, 64), _log(rng, 65, 1024)))
        bias = rng.random() < 0.3
        if kind == "host":
            return dict(kind=kind, fmt=fmt, n=n, k=k, rows=rows, bias=bias)
        return dict(kind=kind, fmt=fmt, n=n, k=k, rows=rows, bias=bias, stack=4 if rows <= 64 else 1)
    hd = rng.choice((64, 128, 128))
    kv = rng.choice((4, 8))
    group = rng.choice((1, 2, 4))
    heads = kv * group
    d = heads * hd if 1024 <= heads * hd <= 4096 else 2048
    shape = dict(layers=rng.randint(2, 16), d=d, heads=heads, kv=kv, hd=hd, ffn=rng.randint(2 * d // 256, 7 * d // 512) * 256,
                 vocab=rng.randint(8000, 64000), mix=rng.choice(sorted(MIX)), interleaved=rng.random() < 0.5)
    if kind == "decode":
        return dict(kind=kind, ctx=_log(rng, 8, 4000), **shape)
    return dict(kind=kind, tokens=_log(rng, 4, 3000), pos0=rng.choice((0, 0, rng.randint(1, 900))), **shape)


# ------------------------------------------------------------------------------------------------- inputs


def _f16(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(-1, 2)


def _quants(gen, nb, count, centre, spread, lo, hi):
    """[nb, count] whole numbers as a quantiser of normal values makes them."""
    q = torch.empty(nb, count, device="cuda").normal_(centre, spread, generator=gen)
    return q.round_().clamp_(lo, hi).to(torch.int16)


def _nibbles(q):
    return (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8)


def _blocks(fmt, nb, gen):
    """nb blocks of the format as one uint8 tensor [nb, bytes], values about N(0, 0.02)."""
    def u(count, lo, hi):
        return torch.empty(nb, count, device="cuda").uniform_(lo, hi, generator=gen)

    def ints(count, lo, hi):
        return torch.randint(lo, hi + 1, (nb, count), device="cuda", generator=gen)

    if fmt == "Q8_0":
        q = _quants(gen, nb, 32, 0.0, 56.0, -127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_f16(u(1, 0.8, 1.2) * (0.02 / 56)), q], 1)
    if fmt == "Q4_0":
        return torch.cat([_f16(u(1, 0.8, 1.2) * (0.02 / 3.5)), _nibbles(_quants(gen, nb, 32, 8.0, 3.5, 0, 15))], 1)
    if fmt == "Q4_1":
        d = u(1, 0.8, 1.2) * (0.02 / 3.5)
        return torch.cat([_f16(d), _f16(-7.5 * d), _nibbles(_quants(gen, nb, 32, 7.5, 3.5, 0, 15))], 1)
    if fmt in ("Q4_K", "Q5_K"):
        centre, spread = (7.5, 3.5) if fmt == "Q4_K" else (15.5, 7.0)
        d = u(1, 0.8, 1.2) * (0.02 / (spread * 52))
        sc, mn = ints(8, 42, 63), ints(8, 42, 63)  # eight 6-bit scales and minima in twelve bytes
        head = torch.cat([(sc[:, :4] | (sc[:, 4:] >> 4 << 6)), (mn[:, :4] | (mn[:, 4:] >> 4 << 6)), (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1).to(torch.uint8)
        parts = [_f16(d), _f16(centre * d), head]
        q = _quants(gen, nb, 256, centre, spread, 0, 15 if fmt == "Q4_K" else 31)
        if fmt == "Q5_K":
            bits = (q >> 4).reshape(nb, 8, 32)
            parts.append(sum(bits[:, i] << i for i in range(8)).to(torch.uint8))
            q = q & 15
        return torch.cat(parts + [_nibbles(q)], 1)
    q = _quants(gen, nb, 256, 32.0, 16.0, 0, 63)  # Q6_K
    hi = (q >> 4).reshape(nb, 4, 64)
    qh = (hi[:, 0] | (hi[:, 1] << 2) | (hi[:, 2] << 4) | (hi[:, 3] << 6)).to(torch.uint8)
    sc = (ints(16, 70, 127) * (2 * ints(16, 0, 1) - 1)).to(torch.int8).view(torch.uint8)
    return torch.cat([_nibbles(q & 15), qh, sc, _f16(u(1, 0.8, 1.2) * (0.02 / (16 * 100)))], 1)


POOL_VALUES = 1 << 24  # (less fifteen blocks: a prime number of them, so that no two rows of a matrix begin alike)


class _Weights:
    """Quantised weights in device memory behind the library's handles: what a user's program keeps for its lifetime.  Each
    matrix is cut from one pool of blocks per format, from a place of its own."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.pools, self.tensors, self.handles = {}, [], []

    def blocks(self, fmt, n, k):
        need = n * (k // BLOCK[fmt][1])
        if fmt not in self.pools:
            self.pools[fmt] = _blocks(fmt, POOL_VALUES // BLOCK[fmt][1] - 15, self.gen)
        pool = self.pools[fmt]
        at = int(torch.randint(0, pool.shape[0], (1,), generator=self.gen, device="cuda").item())
        rolled = torch.cat([pool[at:], pool[:at]])
        return rolled.repeat(-(-need // pool.shape[0]), 1)[:need].contiguous().reshape(-1)

    def add(self, fmt, n, k):
        t = self.blocks(fmt, n, k)
        h = C.c_void_p()
        _lib.check(_lib.lib.jitnn_hip_weight_wrap_dev(BLOCK[fmt][0], C.c_void_p(t.data_ptr()), t.numel(), n, k, C.byref(h)), "jitnn_hip_weight_wrap_dev")
        self.tensors.append(t)
        self.handles.append(h)
        weakref.finalize(t, _lib.lib.jitnn_hip_weight_free, h)
        return h

    def done(self):
        self.pools = {}


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _prepare_model(case, seed, positions):
    w = _Weights(seed)
    d, heads, kv, hd, ffn, vocab, mix = (case[i] for i in ("d", "heads", "kv", "hd", "ffn", "vocab", "mix"))
    model = jitnn_amd.LlamaDecoder(case["layers"], d, heads, kv, hd, ffn, vocab, positions)
    qd, kd = heads * hd, kv * hd
    shapes = ((qd, d), (kd, d), (kd, d), (d, qd), (ffn, d), (ffn, d), (d, ffn), (vocab, d))
    norms = (1.0 + 0.1 * torch.randn(2 * case["layers"] + 1, d, device="cuda", generator=w.gen)).cpu().numpy()
    for layer in range(case["layers"]):
        for which in range(7):
            model.set_weight_handle(layer, which, w.add(MIX[mix][which], *shapes[which]))
        model.set_norm(layer, 0, norms[2 * layer])
        model.set_norm(layer, 1, norms[2 * layer + 1])
    model.set_norm(0, 2, norms[-1])
    model.set_weight_handle(0, 7, w.add(MIX[mix][7], *shapes[7]))
    model.set_rope_interleaved(case["interleaved"])
    return w, model


def _fill_cache(case, w, model, count):
    """`count` positions of keys and values per layer: windows of one N(0, 1) buffer."""
    if count == 0:
        return
    kv = torch.randn(2, count + case["layers"], case["kv"] * case["hd"], device="cuda", generator=w.gen).cpu().numpy()
    for layer in range(case["layers"]):
        model.kv_write(layer, 0, kv[0, layer:layer + count], kv[1, layer:layer + count])


def prepare(case, seed):
    jitnn_amd.init(0)
    kind = case["kind"]
    if kind == "linear":
        w = _Weights(seed)
        n, k, rows = case["n"], case["k"], case["rows"]
        for _ in range(case["stack"]):
            w.add(case["fmt"], n, k)
        w.done()
        return dict(kind=kind, w=w, rows=rows, x=torch.randn(rows, k, device="cuda", generator=w.gen),
                    bias=torch.randn(n, device="cuda", generator=w.gen) if case["bias"] else None,
                    y=[torch.empty(rows, n, device="cuda") for _ in range(case["stack"])])
    if kind == "host":
        w = _Weights(seed)
        n, k = case["n"], case["k"]
        weight = jitnn_amd.Tensor.quantized(jitnn_amd.DType[case["fmt"]], w.blocks(case["fmt"], n, k).cpu().numpy(), n, k)
        x = jitnn_amd.Tensor.of(torch.randn(case["rows"], k, device="cuda", generator=w.gen).cpu().numpy())
        bias = jitnn_amd.Tensor.of(torch.randn(n, device="cuda", generator=w.gen).cpu().numpy()) if case["bias"] else None
        return dict(kind=kind, weight=weight, x=x, bias=bias)
    if kind == "codec":
        w = _Weights(seed)
        n, k = case["n"], case["k"]
        w.add(case["fmt"], n, k)
        w.done()
        return dict(kind=kind, w=w, values=torch.empty(n, k, device="cuda"), q8=torch.empty(n * k // 32 * 34, dtype=torch.uint8, device="cuda"))
    if kind == "decode":
        w, model = _prepare_model(case, seed, case["ctx"] + 1)
        _fill_cache(case, w, model, case["ctx"])
        model.set_embedding(BLOCK["Q4_0"][0], w.blocks("Q4_0", case["vocab"], case["d"]).cpu().numpy())
        w.done()
        token = torch.randint(0, case["vocab"], (1,), device="cuda", generator=w.gen, dtype=torch.int32)
        return dict(kind=kind, w=w, model=model, pos=case["ctx"], token=token, x=torch.empty(case["d"], device="cuda"),
                    logits=torch.empty(case["vocab"], device="cuda"), chosen=torch.empty(1, dtype=torch.int32, device="cuda"))
    w, model = _prepare_model(case, seed, case["pos0"] + case["tokens"])
    _fill_cache(case, w, model, case["pos0"])
    w.done()
    return dict(kind="prefill", w=w, model=model, pos0=case["pos0"], tokens=case["tokens"],
                x=torch.randn(case["tokens"], case["d"], device="cuda", generator=w.gen), logits=torch.empty(case["vocab"], device="cuda"))


# ------------------------------------------------------------------------------------------------- the passes


def run(s):
    lib, check, kind = _lib.lib, _lib.check, s["kind"]
    if kind == "linear":
        x, bias, rows = _ptr(s["x"]), _ptr(s["bias"]), s["rows"]
        for h, y in zip(s["w"].handles, s["y"]):
            check(lib.jitnn_hip_linear_dev(h, x, rows, bias, y.data_ptr(), None), "jitnn_hip_linear_dev")
        return s["y"]
    if kind == "host":
        return jitnn_amd.Gguf.linear(s["x"], s["weight"], s["bias"]).numpy()
    if kind == "codec":
        check(lib.jitnn_hip_dequantize_dev(s["w"].handles[0], _ptr(s["values"]), None), "jitnn_hip_dequantize_dev")
        check(lib.jitnn_hip_quantize_q8_0_dev(_ptr(s["values"]), s["values"].numel(), _ptr(s["q8"]), None), "jitnn_hip_quantize_q8_0_dev")
        return s["values"], s["q8"]
    model, logits = s["model"], s["logits"]
    if kind == "decode":
        check(lib.jitnn_hip_llama_embed_dev(model.handle, _ptr(s["token"]), 1, _ptr(s["x"]), None), "jitnn_hip_llama_embed_dev")
        model.decode_dev(s["x"].data_ptr(), s["pos"], logits.data_ptr())
        check(lib.jitnn_hip_llama_argmax_dev(model.handle, _ptr(logits), _ptr(s["chosen"]), None), "jitnn_hip_llama_argmax_dev")
        return logits, s["chosen"]
    model.prefill_dev(s["x"].data_ptr(), s["pos0"], s["tokens"], logits.data_ptr())
    return logits


# ------------------------------------------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind in ("linear", "host"):
        n, k, rows, stack = case["n"], case["k"], case["rows"], case.get("stack", 1)
        return dict(bytes=4 * rows * k + stack * (nbytes(case["fmt"], n, k) + 4 * rows * n + (4 * n if case["bias"] else 0)), flops=stack * 2 * rows * n * k)
    if kind == "codec":
        n, k = case["n"], case["k"]
        return dict(bytes=nbytes(case["fmt"], n, k) + 4 * n * k + n * k // 32 * 34, flops=0)
    tokens, before = (1, case["ctx"]) if kind == "decode" else (case["tokens"], case["pos0"])
    d, qd, kd, ffn, vocab, layers, mix = case["d"], case["heads"] * case["hd"], case["kv"] * case["hd"], case["ffn"], case["vocab"], case["layers"], MIX[case["mix"]]
    shapes = ((qd, d), (kd, d), (kd, d), (d, qd), (ffn, d), (ffn, d), (d, ffn))
    weights = layers * sum(nbytes(f, n, k) for f, (n, k) in zip(mix, shapes)) + nbytes(mix[7], vocab, d) + 4 * (2 * layers + 1) * d
    cache = layers * 2 * 4 * kd * (before + tokens)  # positions before this pass are read, its own are written
    scores = sum(before + t + 1 for t in range(tokens))
    flops = layers * (2 * tokens * sum(n * k for n, k in shapes) + 4 * qd * scores) + 2 * vocab * d
    return dict(bytes=weights + cache + 4 * (tokens * d + vocab), flops=flops)


def tolerance(case):
    """Relative error (2-norm), four times what was measured.  Linears against FP64 on the dequantised weights: up to 64 rows
    1.4e-7 to 1.8e-6, more rows (FP16 operands) 2.8e-4 to 6.7e-4.  The model at 32 layers: decode, two sets of kernels, 1.3e-5;
    a 40-token prompt against its tokens one by one 1.6e-5; prompts of 512 and 4096 tokens against passes of 64 7e-3.  With
    fewer layers the rounding has less depth to grow over: the square root of their number."""
    kind = case["kind"]
    if kind in ("linear", "host"):
        return {"rel": 7e-6 if case["rows"] <= 64 else 2.6e-3}
    if kind == "codec":
        return "exact"
    depth = math.sqrt(case["layers"] / 32)
    return {"rel": (6e-5 if kind == "decode" or case["tokens"] <= 64 else 3e-2) * depth}
