"""The attention of long prompts on packed keys and values: by itself (tests/attention_packed_test.hip, built with the library) against
FP64, and as a prompt pass takes it, against the same tokens in passes too short for it."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

from helpers import random_valid_blocks

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent
PROGRAM = ROOT / "tests" / "build" / "attention_packed_test"


def test_attention_packed():
    if not PROGRAM.exists():
        subprocess.run(["make", "-C", str(ROOT / "jitnn_amd" / "csrc"), "tests"], check=True)
    done = subprocess.run([str(PROGRAM)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout.endswith("all hold\n"), done.stdout + done.stderr


@pytest.mark.parametrize("heads,kv,hd,pos0,tokens", [(32, 8, 64, 3, 2050), (16, 16, 128, 130, 4097), (48, 3, 64, 0, 1401)])
def test_prompt_pass(heads, kv, hd, pos0, tokens):
    """One layer whose prompt is 384 to 526 workgroups of 128 rows, in one pass and in passes of 256 tokens (16 to 128 workgroups, the
    former kernel).  Every operand of both is rounded to FP16 the same way and summed in FP32; what differs is the order of the sums and
    where a row's running maximum stands when a weight is rounded, 2^-11 of each weight: 2^-10 of the values' magnitude, through the
    projections behind the attention 3e-3 of the logits' (2-norm)."""
    import jitnn_amd
    import torch
    jitnn_amd.init()
    d, ffn, vocab = 256, 256, 512
    rng = np.random.default_rng(tokens)
    shapes = ((heads * hd, d), (kv * hd, d), (kv * hd, d), (d, heads * hd), (ffn, d), (ffn, d), (d, ffn), (vocab, d))
    weights = [jitnn_amd.Tensor.quantized(jitnn_amd.DType.Q8_0, random_valid_blocks(rng, "Q8_0", n, k), n, k) for n, k in shapes]
    x = torch.randn(pos0 + tokens, d, device="cuda", generator=torch.Generator(device="cuda").manual_seed(heads))
    out = []
    for step in (tokens, 256):
        model = jitnn_amd.LlamaDecoder(1, d, heads, kv, hd, ffn, vocab, pos0 + tokens)
        for i, w in enumerate(weights):
            model.set_weight_handle(0, i, w.handle)
        for which in range(3):
            model.set_norm(0, which, np.ones(d, np.float32))
        logits = torch.empty(vocab, device="cuda")
        if pos0:
            model.prefill_dev(x.data_ptr(), 0, pos0, None)
        for t in range(0, tokens, step):
            model.prefill_dev(x[pos0 + t:].data_ptr(), pos0 + t, min(step, tokens - t), logits.data_ptr())
        torch.cuda.synchronize()
        out.append(logits.cpu().double().numpy())
        model.close()
    assert np.isfinite(out[0]).all()
    assert np.linalg.norm(out[0] - out[1]) <= 3e-3 * np.linalg.norm(out[1])
