"""The attention of long prompts on the matrix cores against the same prompt in pieces of 400 tokens, which take 64 query rows per
workgroup: 128 rows per workgroup (attn_prefill_mfma_kernel<D, 2>: from one workgroup per CU on for heads of 128 values, two for 64), where
every row meets the same chunks of keys in the same order with the same FP16 operands and FP32 sums, and the kernel on packed
keys and values, with queries of 22 bits and a running maximum per 64 keys.  Which one ran is asserted.  What differs besides is the route
of the linears (FP16 operands, K cut elsewhere).  The second layer's keys and values follow from the attention output of every
token of the first.

Tolerance: two sets of FP16-operand linears, 2e-3 of the largest magnitude each (a wrong row of the attention is off by 1e-1)."""
import numpy as np
import pytest

from helpers import norm_err
from test_gpu_decode import SLOTS, build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,head_dim,tokens,pos0,packing,how", [
    (32, 8, 64, 2060, 5, False, "MFMA_128"), (32, 8, 64, 2060, 5, True, "PACKED"),  # groups of four; the last block partly filled, keys in front of the prompt
    (32, 8, 128, 1090, 0, False, "MFMA_128"), (32, 8, 128, 1090, 0, True, "PACKED"),
    (24, 8, 64, 2700, 63, False, "MFMA_128"), (24, 8, 64, 2700, 63, True, "PACKED"),  # groups of three: 126 of a block's 128 rows, and the mask on every chunk
    (8, 8, 128, 4000, 1, False, "MFMA_128"), (8, 8, 128, 4000, 1, True, "PACKED"),  # one query head per key / value head
    (20, 4, 64, 3300, 0, False, "MFMA_128"), (20, 4, 64, 3300, 0, True, "PACKED"),  # groups of five over four heads
    (32, 8, 64, 1030, 5, True, "MFMA_64"), (24, 8, 64, 1400, 63, False, "MFMA_64"), (10, 2, 64, 3300, 0, True, "MFMA_64")])  # (too few workgroups for either)
def test_long_prompt_in_one_pass_and_in_pieces(heads, kv_heads, head_dim, tokens, pos0, packing, how):
    import jitnn_amd as jn
    from jitnn_amd import _lib
    jn.init()
    d = 512
    cfg = dict(layers=2, d_model=d, heads=heads, kv_heads=kv_heads, head_dim=head_dim, ffn=512, vocab=300, max_ctx=pos0 + tokens, rms_eps=1e-5, rope_theta=5e5)
    dec, _, _, _ = build(jn, cfg, 29, {s: "Q8_0" for s in SLOTS}, "Q8_0")
    dec.set_packing(packing)
    rng = np.random.default_rng(heads + tokens)
    x = rng.standard_normal((pos0 + tokens, d)).astype(np.float32)
    if pos0:
        dec.prefill(x[:pos0], 0)
    whole = dec.prefill(x[pos0:], pos0)
    assert dec.last_attention() == getattr(_lib, "ATTN_" + how)
    got = dec.kv_read(1, pos0, tokens)
    for at in range(pos0, pos0 + tokens, 400):
        pieces = dec.prefill(x[at:min(at + 400, pos0 + tokens)], at)
        assert dec.last_attention() in (_lib.ATTN_MFMA_64, _lib.ATTN_FP32)  # (the last piece may be 64 tokens or fewer)
    ref = dec.kv_read(1, pos0, tokens)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert norm_err(a, b) <= 4e-3
    assert norm_err(whole, pieces) <= 4e-3
    dec.close()
