"""The attention of long prompts on packed keys and values: by itself (tests/attention_packed_test.hip, built with the library) against
FP64, as a prompt pass takes it, against the same tokens in passes too short for it, and a pass that cannot have its buffer."""
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

from decode_oracle import SLOTS
from helpers import norm_err
from test_gpu_decode import build

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent
PROGRAM = ROOT / "tests" / "build" / "attention_packed_test"


def test_attention_packed():
    if not PROGRAM.exists():
        subprocess.run(["make", "-C", str(ROOT / "jitnn_amd" / "csrc"), "tests"], check=True)
    done = subprocess.run([str(PROGRAM)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout.endswith("all hold\n"), done.stdout + done.stderr


def model(heads, kv, hd, positions, seed):
    """Two layers with scores a few units wide: the norms in front of q, k and v are six times as large as elsewhere."""
    import jitnn_amd as jn
    jn.init()
    cfg = dict(layers=2, d_model=256, heads=heads, kv_heads=kv, head_dim=hd, ffn=256, vocab=512, max_ctx=positions, rms_eps=1e-5, rope_theta=5e5)
    dec = build(jn, cfg, seed, {s: "Q8_0" for s in SLOTS}, "Q8_0")[0]
    for layer in range(2):
        dec.set_norm(layer, 0, np.full(256, 6, np.float32))
    return dec


@pytest.mark.parametrize("heads,kv,hd,pos0,tokens", [(32, 8, 64, 3, 2050), (16, 16, 128, 130, 4097), (48, 3, 64, 0, 1401)])
def test_prompt_pass(heads, kv, hd, pos0, tokens):
    """A prompt of 520 to 528 workgroups of 128 rows on packed keys and values, and the same in passes of 256 tokens (32 to 96
    workgroups: 64 query rows each, keys and values as they are).  The second layer's keys and values follow from the attention output of
    every token of the first.  Keys, values and weights are rounded to FP16 in both, 2^-11 each; the queries are here to 22 bits and there
    to 11: scores a few units wide, 2^-9 of a weight at most, through the projections behind the attention 4e-3 of the largest magnitude."""
    from jitnn_amd import _lib
    dec = model(heads, kv, hd, pos0 + tokens, heads)
    x = np.random.default_rng(tokens).standard_normal((pos0 + tokens, 256)).astype(np.float32)
    if pos0:
        dec.prefill(x[:pos0], 0, logits=False)
    out = [dec.prefill(x[pos0:], pos0), *dec.kv_read(1, pos0, tokens)]
    assert dec.last_attention() == _lib.ATTN_PACKED
    for at in range(pos0, pos0 + tokens, 256):
        last = dec.prefill(x[at:min(at + 256, pos0 + tokens)], at)
        assert dec.last_attention() in (_lib.ATTN_MFMA_64, _lib.ATTN_FP32)
    for a, b in zip(out, [last, *dec.kv_read(1, pos0, tokens)]):
        assert np.isfinite(a).all()
        assert norm_err(a, b) <= 4e-3
    dec.close()


def test_without_room_under_a_capture_and_with_it_again():
    """A pass that is recorded before any eager pass wanted the packed copy takes the kernel of 64 query rows, with the bits of a model that
    does without; the next eager pass asks for the room again."""
    from jitnn_amd import _lib
    heads, kv, hd, tokens, pos0 = 32, 8, 128, 600, 900  # 152 workgroups of 128 rows: packed behind 900 positions, not from position 0
    dec = model(heads, kv, hd, pos0 + tokens, 7)
    x = torch.randn(pos0 + tokens, 256, device="cuda", generator=torch.Generator(device="cuda").manual_seed(7))

    def run(at, count, stream, logits):
        dec.prefill_dev(x[at:].data_ptr(), at, count, logits.data_ptr(), stream.cuda_stream)

    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    logits, ref = torch.empty(512, device="cuda"), torch.empty(512, device="cuda")
    with torch.cuda.stream(side):
        for at in (0, 300):  # (the buffers of 600 tokens, and the positions in front)
            run(at, tokens, side, logits)
            assert dec.last_attention() == _lib.ATTN_MFMA_64
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            run(pos0, tokens, side, logits)
        assert dec.last_attention() == _lib.ATTN_MFMA_64
        dec.set_packing(False)
        run(pos0, tokens, side, ref)
        assert dec.last_attention() == _lib.ATTN_MFMA_64
        side.synchronize()
        for _ in range(3):
            logits.fill_(float("nan"))
            graph.replay()
            side.synchronize()
            assert torch.equal(logits, ref)
        dec.set_packing(True)
        run(pos0, tokens, side, logits)
        assert dec.last_attention() == _lib.ATTN_PACKED
        side.synchronize()
        assert (logits - ref).abs().max() <= 4e-3 * ref.abs().max()
    del graph
    dec.close()
