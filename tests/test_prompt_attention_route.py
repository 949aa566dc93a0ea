"""Which kernel the attention of a prompt pass takes, asked of the library without a device, for 256 compute units: both sides of every line of
the rule, where it was measured (us per layer of whole prompts beside attn_packed_pays)."""
import pytest

FP32, DOT2, MFMA_64, MFMA_128, PACKED = range(5)


@pytest.mark.parametrize("heads,kv,hd,pos0,tokens,how,without", [
    (32, 8, 128, 0, 64, FP32, FP32), (32, 8, 64, 900, 64, FP32, FP32), (8, 8, 192, 0, 65, DOT2, DOT2), (16, 1, 256, 0, 4096, DOT2, DOT2),
    (32, 8, 128, 0, 65, MFMA_64, MFMA_64), (32, 8, 128, 0, 672, MFMA_64, MFMA_64), (32, 8, 128, 0, 673, PACKED, MFMA_64),  # 168 and 176 blocks
    (32, 8, 128, 0, 992, PACKED, MFMA_64), (32, 8, 128, 0, 993, PACKED, MFMA_128),  # 248 and 256
    (32, 8, 128, 900, 600, PACKED, MFMA_64), (16, 4, 128, 900, 1200, PACKED, MFMA_64), (16, 4, 128, 899, 1200, MFMA_64, MFMA_64),
    (8, 4, 128, 900, 2200, MFMA_64, MFMA_64), (32, 8, 128, 2000, 512, MFMA_64, MFMA_64), (32, 8, 128, 2000, 513, PACKED, MFMA_64),  # 128 and 136
    (32, 8, 64, 0, 1248, MFMA_64, MFMA_64), (32, 8, 64, 0, 1249, PACKED, MFMA_64),  # 312 and 320
    (32, 8, 64, 5000, 1248, MFMA_64, MFMA_64), (32, 8, 64, 0, 2016, PACKED, MFMA_64), (32, 8, 64, 0, 2017, PACKED, MFMA_128)])  # 504 and 512
def test_route(heads, kv, hd, pos0, tokens, how, without):
    from jitnn_amd._lib import prompt_attention
    assert prompt_attention(heads, kv, hd, pos0, tokens, compute_units=256) == how
    assert prompt_attention(heads, kv, hd, pos0, tokens, packing=False, compute_units=256) == without


@pytest.mark.parametrize("hd", [64, 128])
def test_a_heads_packed_keys_stay_below_two_gib(hd):
    """The kernel reaches a head's chunks by 32-bit offsets into one buffer descriptor: 4 bytes per position and value, 2 GiB less a chunk."""
    from jitnn_amd._lib import prompt_attention
    most = (1 << 31) // (4 * hd) - 64
    for keys, how in ((most, PACKED), (most + 1, MFMA_128), (2 * most, MFMA_128), (1 << 30, MFMA_128)):
        assert prompt_attention(8, 8, hd, keys - 9000, 9000, compute_units=256) == how


def test_misuse():
    from jitnn_amd._lib import prompt_attention
    for heads, kv, hd, pos0, tokens, cus in ((7, 2, 128, 0, 100, 256), (34, 2, 128, 0, 100, 256), (8, 8, 96, 0, 100, 256), (8, 8, 128, -1, 100, 256),
                                             (8, 8, 128, 0, 0, 256), (8, 8, 128, (1 << 31) - 100, 100, 256), (8, 8, 128, 0, 100, -1)):
        with pytest.raises(ValueError):
            prompt_attention(heads, kv, hd, pos0, tokens, compute_units=cus)
