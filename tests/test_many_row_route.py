"""Which of the two kernels for more than 64 rows a launch takes (wide_pays / wide_plan in jitnn_hip.hip), asked of the library
without a device, for 256 compute units."""
import pytest

from helpers import GGML_ID

# the launches of a layer of the Llama-8B shape (Q4_K, v and down Q6_K): tokens -> weight rows per tile of (q, k and v; attn_o with the
# residual; gate and up as one product; down with the residual), 0: the kernel that decodes as it goes
# (the table moves with the figures of the rule; it says which launches a test of a given length reaches)
LAYER = [(65, (0, 0, 0, 0)),
         (512, (0, 0, 0, 0)),
         (513, (0, 0, 0, 0)),
         (1024, (0, 0, 0, 0)),
         (1025, (0, 0, 0, 128)),
         (1280, (0, 0, 0, 128)),
         (1281, (192, 0, 0, 128)),
         (1792, (192, 0, 0, 128)),
         (1793, (256, 0, 0, 128)),
         (1874, (256, 0, 0, 128)),
         (1875, (256, 128, 0, 128)),
         (2048, (256, 128, 0, 128)),
         (2049, (256, 192, 256, 192)),
         (2304, (256, 192, 256, 192)),
         (2305, (256, 192, 0, 192)),
         (2560, (256, 192, 0, 192)),
         (2561, (192, 192, 256, 192)),
         (2816, (192, 192, 256, 192)),
         (2817, (192, 256, 0, 256)),
         (3072, (192, 256, 0, 256)),
         (3073, (192, 256, 256, 256)),
         (3328, (192, 256, 256, 256)),
         (3329, (192, 256, 0, 256)),
         (3584, (192, 256, 0, 256)),
         (3585, (192, 256, 256, 256)),
         (3840, (192, 256, 256, 256)),
         (3841, (128, 256, 256, 256)),
         (4096, (128, 256, 256, 256))]


@pytest.mark.parametrize("tokens,tiles", LAYER)
def test_layer_of_the_8b_shape(tokens, tiles):
    from jitnn_amd._lib import many_row_tile
    k4, k6 = GGML_ID["Q4_K"], GGML_ID["Q6_K"]
    got = (many_row_tile([(k4, 4096), (k4, 1024), (k6, 1024)], 4096, tokens, compute_units=256),
           many_row_tile([(k4, 4096)], 4096, tokens, residual=True, compute_units=256),
           many_row_tile([(k4, 14336), (k4, 14336)], 4096, tokens, gate_up=True, compute_units=256),
           many_row_tile([(k6, 4096)], 14336, tokens, residual=True, compute_units=256))
    assert got == tiles


@pytest.mark.parametrize("fmt,n,k,rows,tile", [
    ("Q4_0", 11003, 1056, 512, 0), ("Q4_0", 11003, 1056, 513, 192),      # more than two tiles of tokens
    ("Q4_0", 11003, 1023 // 32 * 32, 2000, 0), ("Q4_0", 11003, 1024, 2000, 192),  # rows of at least 1024 values
    ("Q8_0", 1024, 4096, 1024, 0),                                       # splits K
    ("Q5_0", 11003, 1056, 2000, 0),                                      # no many-row kernel
    ("Q4_K", 128256, 4096, 4096, 0)])                                    # more than 512 MiB of dequantised weights
def test_edges_of_the_rule(fmt, n, k, rows, tile):
    from jitnn_amd._lib import many_row_tile
    assert many_row_tile([(GGML_ID[fmt], n)], k, rows, compute_units=256) == tile


def test_misuse():
    from jitnn_amd._lib import many_row_tile
    k4 = GGML_ID["Q4_K"]
    for weights, k, kw in (([(k4, 64)], 100, {}), ([(99, 64)], 256, {}), ([(k4, 64), (k4, 32)], 256, dict(gate_up=True)),
                           ([(k4, 64), (k4, 64)], 256, dict(residual=True)), ([(k4, 64)] * 4, 256, {})):
        with pytest.raises(ValueError):
            many_row_tile(weights, k, 2000, compute_units=256, **kw)


@pytest.mark.parametrize("fmt,n,k,rows,tile", [
    ("Q4_0", 14336, 4096, 512, 0), ("Q4_0", 14336, 4096, 900, 0), ("Q4_1", 14336, 4096, 900, 0), ("Q5_K", 14336, 4096, 900, 0),
    ("Q8_0", 14336, 4096, 900, 256), ("Q4_0", 4352, 12800, 886, 0), ("Q4_0", 14336, 4096, 1024, 0), ("Q4_0", 4096, 14336, 2048, 128), ("Q8_0", 4352, 12800, 886, 128)])
def test_formats_decoded_in_packed_fp16(fmt, n, k, rows, tile):
    """Up to 1024 rows Q4_0, Q4_1 and Q5_K stay with the kernel that decodes as it goes where Q8_0, whose decode is longer, does not."""
    from jitnn_amd._lib import many_row_tile
    assert many_row_tile([(GGML_ID[fmt], n)], k, rows, compute_units=256) == tile
