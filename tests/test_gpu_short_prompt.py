"""Prompts of 9 to 64 tokens through layers whose rows are longer than 2048 values, so that linears come in slices of a row that the
next kernel adds up: q, k and v in the rotation, attn_o and ffn_down in the RMSNorm, gate and up in the preparation of ffn_down's
operands - or, where q, k and v do not fit the buffer lent for it, in a launch of their own.  Two layers against the oracle: the last
token's logits and the keys and values of the second layer, which follow from every token's output of the first.

Tolerance: 2e-6 of the largest output per linear (two FP16 parts of an operand, FP32 sums) and nine of them in a row from the input to
the logits: 2e-5 of the largest magnitude."""
import numpy as np
import pytest
import torch

from decode_oracle import prefill_ref
from helpers import GGML_ID, norm_err
from test_gpu_decode import MIX, SLOTS, build

pytestmark = pytest.mark.gpu

Q5_K_M = {**dict.fromkeys(SLOTS, "Q5_K"), "attn_v": "Q6_K", "ffn_down": "Q6_K"}
Q6_K = dict.fromkeys(SLOTS, "Q6_K")


def slices(cfg, mix, tokens):
    """Slices of every linear of a layer, 0: it has none.  (A launch that others join is cheaper than one that joins: no fewer
    come in slices in the prompt pass.)"""
    from jitnn_amd._lib import few_rows_slices
    d, qd, kd, ffn = cfg["d_model"], cfg["heads"] * cfg["head_dim"], cfg["kv_heads"] * cfg["head_dim"], cfg["ffn"]
    shapes = {"attn_q": (qd, d), "attn_k": (kd, d), "attn_v": (kd, d), "attn_o": (d, qd), "ffn_gate": (ffn, d), "ffn_up": (ffn, d), "ffn_down": (d, ffn)}
    return tuple(few_rows_slices(GGML_ID[mix[s]], *shapes[s], tokens, adds=s in ("attn_o", "ffn_down")) for s in SLOTS)


@pytest.fixture(scope="module")
def jn():
    import jitnn_amd
    jitnn_amd.init()
    return jitnn_amd


# per prompt: tokens, position, slices of q, k, v, o, gate, up, down, floats in front of the input (1: not aligned to 16 bytes)
@pytest.mark.parametrize("mix,ffn,interleaved,prompts", [
    (MIX, 7168, False, [(9, 37, (0, 0, 2, 0, 2, 2, 4), 0), (40, 0, (2, 0, 2, 2, 2, 2, 4), 0), (40, 0, (2, 0, 2, 2, 2, 2, 4), 1), (64, 3, (2, 0, 2, 2, 2, 2, 4), 3)]),
    (Q6_K, 14336, True, [(9, 0, (2, 2, 2, 2, 2, 2, 7), 0), (57, 20, (2, 2, 2, 2, 0, 0, 7), 0)]),
    (Q5_K_M, 2560, False, [(24, 11, (0, 0, 2, 0, 0, 0, 2), 0), (64, 0, (2, 0, 2, 2, 2, 2, 2), 1)])], ids=["q4_k_m", "q6_k", "q5_k_m"])
def test_short_prompt_with_long_rows(jn, mix, ffn, interleaved, prompts):
    cfg = dict(layers=2, d_model=2304, heads=20, kv_heads=4, head_dim=128, ffn=ffn, vocab=300, max_ctx=80, rms_eps=1e-5, rope_theta=1e4)
    dec, layers, out_norm, out_w = build(jn, cfg, 13, mix, "Q6_K")
    dec.set_rope_interleaved(interleaved)
    rng = np.random.default_rng(ffn)
    for tokens, pos0, want, off in prompts:
        assert slices(cfg, mix, tokens) == want
        kc, vc = (np.zeros((2, 80, 4, 128), dtype=np.float32) for _ in range(2))
        kc[:, :pos0], vc[:, :pos0] = rng.standard_normal((2, 2, pos0, 4, 128))
        for li in range(2 if pos0 else 0):
            dec.kv_write(li, 0, kc[li, :pos0], vc[li, :pos0])
        x = rng.standard_normal((tokens, 2304)).astype(np.float32)
        buf = torch.zeros(off + x.size, device="cuda")
        buf[off:] = torch.from_numpy(x).reshape(-1).cuda()
        logits = torch.full((300,), float("nan"), device="cuda")
        assert buf.data_ptr() % 16 == 0
        torch.cuda.synchronize()
        dec.prefill_dev(buf.data_ptr() + 4 * off, pos0, tokens, logits.data_ptr())
        torch.cuda.synchronize()
        check(dec, cfg, layers, out_norm, out_w, kc, vc, x, pos0, logits.cpu().numpy(), interleaved)
    dec.close()


def check(dec, cfg, layers, out_norm, out_w, kc, vc, x, pos0, logits, interleaved=False):
    ref = prefill_ref(cfg, layers, out_norm, out_w, kc, vc, x, pos0, interleaved)
    errs = [norm_err(logits, ref)]
    for li in range(2):
        k, v = dec.kv_read(li, pos0, len(x))
        errs += [norm_err(k, kc[li, pos0:pos0 + len(x)]), norm_err(v, vc[li, pos0:pos0 + len(x)])]
    assert max(errs) <= 2e-5, (len(x), pos0, errs)


@pytest.mark.parametrize("heads,kv_heads,head_dim,tokens,o_slices", [(128, 8, 64, 64, 4), (128, 8, 128, 40, 8), (80, 5, 64, 64, 3)])
def test_short_prompt_with_many_heads(jn, heads, kv_heads, head_dim, tokens, o_slices):
    """More than half as many blocks of 32 query rows as compute units: the attention of short prompts in such blocks, where a prompt on fewer heads
    takes blocks of 16; and attn_o in up to eight slices, the most the norm adds up.  Groups of sixteen, keys in front of the prompt."""
    cfg = dict(layers=2, d_model=512, heads=heads, kv_heads=kv_heads, head_dim=head_dim, ffn=512, vocab=200, max_ctx=75, rms_eps=1e-5, rope_theta=1e4)
    assert 2 * -(-tokens // (32 // (heads // kv_heads))) * kv_heads > jn.device_info()["compute_units"]
    assert slices(cfg, Q6_K, tokens)[3] == o_slices
    dec, layers, out_norm, out_w = build(jn, cfg, 17, Q6_K, "Q6_K")
    rng = np.random.default_rng(heads)
    kc, vc = (np.zeros((2, 75, kv_heads, head_dim), dtype=np.float32) for _ in range(2))
    kc[:, :11], vc[:, :11] = rng.standard_normal((2, 2, 11, kv_heads, head_dim))
    for li in range(2):
        dec.kv_write(li, 0, kc[li, :11], vc[li, :11])
    x = rng.standard_normal((tokens, 512)).astype(np.float32)
    check(dec, cfg, layers, out_norm, out_w, kc, vc, x, 11, dec.prefill(x, 11))
    dec.close()
