"""The decode step's attention over a long cache: the kernel by itself (tests/attention_split_test.hip, built with the library) against
FP64, and as a decode step takes it, against the oracle's composition of the reference operators."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

from decode_oracle import SLOTS, decode_ref
from helpers import norm_err
from test_gpu_decode import build

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent
PROGRAM = ROOT / "tests" / "build" / "attention_split_test"


def test_attention_split():
    if not PROGRAM.exists():
        subprocess.run(["make", "-C", str(ROOT / "jitnn_amd" / "csrc"), "tests"], check=True)
    done = subprocess.run([str(PROGRAM)], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.endswith("all hold\n"), done.stdout[-2000:] + done.stderr


@pytest.mark.parametrize("heads,kv,hd,ctx,interleaved", [(8, 8, 128, 1022, False), (6, 2, 64, 1023, True), (4, 4, 64, 4090, False), (32, 8, 128, 2303, True)])
def test_decode_step(heads, kv, hd, ctx, interleaved):
    """Four tokens in a row, from the last position of the kernel for short caches, or across the end of a chunk."""
    import jitnn_amd as jn
    jn.init()
    cfg = dict(layers=1, d_model=256, heads=heads, kv_heads=kv, head_dim=hd, ffn=256, vocab=100, max_ctx=ctx + 4, rms_eps=1e-5, rope_theta=5e5)
    dec, layers, out_norm, out_w = build(jn, cfg, 17, {s: "Q8_0" for s in SLOTS}, "Q8_0")
    dec.set_rope_interleaved(interleaved)
    rng = np.random.default_rng(ctx)
    kc = np.zeros((1, cfg["max_ctx"], kv, hd), dtype=np.float32)
    vc = np.zeros_like(kc)
    kc[:, :ctx] = rng.standard_normal(kc[:, :ctx].shape)
    vc[:, :ctx] = rng.standard_normal(vc[:, :ctx].shape)
    dec.kv_write(0, 0, kc[0, :ctx], vc[0, :ctx])
    for pos in range(ctx, ctx + 4):
        x = rng.standard_normal(cfg["d_model"]).astype(np.float32)
        ref = decode_ref(cfg, layers, out_norm, out_w, kc, vc, x, pos, rope_interleaved=interleaved)
        assert norm_err(dec.decode(x, pos), ref) <= 1e-4, pos
        k, v = dec.kv_read(0, pos, 1)
        assert np.allclose(k[0], kc[0, pos], rtol=1e-5, atol=1e-6) and np.allclose(v[0], vc[0, pos], rtol=1e-5, atol=1e-6)
    dec.close()
