"""The dequantiser's streamed stores (outputs beyond 192 MiB) beside its plain ones, on the device: the largest output that is stored
plainly and the smallest that is streamed, the same bits as the oracle's, and the Q8_0 quantiser reading them from there in stream order."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import GGML_ID, random_valid_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("fmt", ["Q4_0", "Q5_1", "Q8_0", "Q4_K", "Q6_K"])
def test_dequantised_on_the_device_then_quantised(fmt, extra):
    import jitnn_amd
    from jitnn_amd import _lib
    from oracle import oracle
    jitnn_amd.init()
    n, k = (192 << 18) // 256 + extra, 256
    raw = random_valid_blocks(np.random.default_rng(n), fmt, n, k)
    w = jitnn_amd.Tensor.quantized(jitnn_amd.DType[fmt], raw, n, k)
    y = torch.full((n * k + 4,), -7.0, device="cuda")
    q = torch.full((n * k // 32 * 34 + 4,), 77, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.lib.jitnn_hip_dequantize_dev(w.handle, C.c_void_p(y.data_ptr()), None), "jitnn_hip_dequantize_dev")
    _lib.check(_lib.lib.jitnn_hip_quantize_q8_0_dev(C.c_void_p(y.data_ptr()), n * k, C.c_void_p(q.data_ptr()), None), "jitnn_hip_quantize_q8_0_dev")
    torch.cuda.synchronize()
    ref = oracle.dequantize(GGML_ID[fmt], raw, n * k)
    assert np.array_equal(y[:n * k].cpu().numpy().view(np.uint32), ref.view(np.uint32)) and (y[n * k:] == -7.0).all()
    assert np.array_equal(q[:-4].cpu().numpy(), oracle.quantize_q8_0(ref)) and (q[-4:] == 77).all()
