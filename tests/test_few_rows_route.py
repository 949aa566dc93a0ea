"""Which of the two kernels for 9 to 64 rows a linear takes (gemv_held_plan in gemv_rows.hip), asked of the library without a
device, for 256 compute units: launches where one kernel was measured at least four per cent ahead of the other.  The comments are
us with the streaming kernel / the held one (profiles/linears_9_to_64_rows_both_kernels.txt)."""
import pytest

from helpers import GGML_ID


@pytest.mark.parametrize("fmt,n,k,rows", [
    ("Q5_1", 1792, 8448, 44),   # 20.7 / 24.3
    ("Q5_1", 5000, 2816, 9),    # 15.8 / 17.1
    ("Q5_1", 25486, 2304, 48),  # 56.6 / 61.6
    ("Q5_1", 14336, 4096, 40),  # 35.3 / 36.8
    ("Q4_1", 4096, 8192, 40),   # 23.7 / 25.2
    ("Q4_0", 2048, 11264, 40),  # 23.0 / 25.2
    ("Q4_0", 6400, 3584, 33),   # 24.4 / 26.9
    ("Q8_0", 13312, 4352, 48),  # 45.2 / 49.2
    ("Q8_0", 2000, 6912, 40)])  # 19.2 / 20.1
def test_streaming_where_the_held_kernel_is_slower(fmt, n, k, rows):
    from jitnn_amd._lib import few_rows_slices
    assert few_rows_slices(GGML_ID[fmt], n, k, rows, compute_units=256) == 0


@pytest.mark.parametrize("fmt,n,k,rows,slices", [
    ("Q6_K", 4096, 14336, 40, 7),  # 49.8 / 44.3
    ("Q6_K", 512, 11008, 12, 6),   # 27.8 / 15.0
    ("Q6_K", 4096, 14336, 8, 7),   # 33.3 / 30.9
    ("Q4_K", 14336, 4096, 24, 2),  # 25.3 / 23.6
    ("Q4_K", 5000, 2816, 40, 2),   # 23.5 / 19.5
    ("Q5_K", 4096, 14336, 24, 7),  # 32.2 / 27.4
    ("Q5_K", 5000, 2816, 40, 2),   # 24.2 / 20.6
    ("Q4_0", 24000, 2048, 24, 1),  # 26.4 / 23.3
    ("Q4_1", 4096, 14336, 24, 7),  # 31.0 / 26.9
    ("Q5_1", 24000, 2048, 24, 1),  # 26.8 / 24.5
    ("Q2_K", 4096, 14336, 40, 7)])  # 40.4 / 31.3
def test_held_where_it_is_faster(fmt, n, k, rows, slices):
    from jitnn_amd._lib import few_rows_slices
    assert few_rows_slices(GGML_ID[fmt], n, k, rows, compute_units=256) == slices


@pytest.mark.parametrize("fmt,n,k,rows", [("Q6_K", 4096, 14336, 65), ("Q6_K", 4096, 14336, 2), ("Q6_K", 4096, 8192, 8), ("Q6_K", 15, 14336, 40),
                                          ("Q8_0", 4096, 14336 + 32, 40), ("Q4_0", 4096, 4096, 11), ("Q5_0", 4096, 14336, 40)])
def test_launches_of_other_kernels(fmt, n, k, rows):
    from jitnn_amd._lib import few_rows_slices
    assert few_rows_slices(GGML_ID[fmt], n, k, rows, compute_units=256) == 0


def test_misuse():
    from jitnn_amd._lib import few_rows_slices
    for fmt, n, k, rows, cus in ((12, 64, 100, 16, 256), (99, 64, 256, 16, 256), (12, 64, 256, 0, 256), (12, 64, 256, 16, -1)):
        with pytest.raises(ValueError):
            few_rows_slices(fmt, n, k, rows, compute_units=cus)
