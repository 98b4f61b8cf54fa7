"""Which kernel a linear layer of few rows goes to: the rules have no GPU in
them. Sizes at which one way was measured well ahead, weights that no cache
holds; us of the library, of the streaming kernels and of one row of tiles."""

import pytest

import fusioninfer_amd.ops as ops

pytestmark = pytest.mark.skipif(ops._C is None, reason="extension not built")


def way(rows, n, k, silu_mul=False):
    if not ops._streams(rows, n, k, silu_mul):
        return "library"
    if rows > 128 and ops._one_row(rows, n, k, silu_mul):
        return "tiles"
    return "streams"


@pytest.mark.parametrize("rows,n,k,want", [
    (144, 8192, 2048, "library"),      # 15.8, 21.5
    (160, 3072, 4096, "library"),      # 16.7, 20.9
    (160, 57344, 8192, "library"),     # 183, 223
    (256, 57344, 9728, "library"),     # 253, 312
    (256, 40960, 4096, "library"),     # 93, 110, 107
    (256, 4096, 2048, "library"),      # 13.7, 20.2
    (144, 16384, 2560, "library"),     # 28.6, 32.9
    (144, 6144, 4096, "streams"),      # 39.6, 24.4
    (160, 4096, 4096, "streams"),      # 27.2, 21.6
    (192, 4096, 4096, "streams"),      # 33.2, 22.7
    (256, 6144, 4096, "streams"),      # 40.0, 30.1
    (256, 8192, 8192, "streams"),      # 75, 52
    (64, 4096, 12288, "streams"),      # 36.7, 26.1
    (128, 4096, 12288, "streams"),     # 66.2, 32.7
    (256, 151936, 4096, "tiles"),      # 361, 343, 303
    (192, 65536, 2048, "tiles"),       # 76, 69, 60
    (160, 28672, 1024, "library"),     # 18.8, 19.5
])
def test_choice(rows, n, k, want):
    assert way(rows, n, k) == want


@pytest.mark.parametrize("rows,n,k,want", [
    (160, 57344, 8192, "library"),
    (256, 24576, 4096, "streams"),     # 72, 58.7
    (256, 40960, 2048, "tiles"),
    (256, 28672, 4096, "streams"),
])
def test_choice_with_silu(rows, n, k, want):
    assert way(rows, n, k, True) == want


@pytest.mark.parametrize("rows,n,k,want", [
    (16, 24576, 4096, True),      # 30.0, 19.3
    (43, 2560, 4096, False),      # 8.9, 10.6
    (64, 4096, 12288, True),      # 24.2, 18.0
    (64, 7168, 8192, False),      # 18.1, 21.7
    (96, 4096, 12288, True),      # 29.9, 23.9
    (128, 6144, 4096, False),     # 15.6, 19.4
])
def test_choice_e4m3(rows, n, k, want):
    assert ops._streams_fp8(rows, n, k) == want


@pytest.mark.parametrize("rows,n,k,want", [
    (17, 6144, 4096, True), (128, 6144, 4096, True),   # 26.5 apart, 25.6
    (64, 5120, 8192, True), (64, 5120, 12288, False),
    (65, 5120, 8192, False),      # 29.3, 31.2
    (128, 8192, 4096, False),     # 28.3, 29.1
    (64, 10240, 4096, True), (65, 10240, 4096, False),   # 29.1, 31.4
])
def test_choice_of_heads_from_pieces(rows, n, k, want):
    assert ops._rope_in_one(rows, n, k) == want


def test_estimates_grow():
    """With either size of W, whatever the shape of a tile is."""
    for rows in (17, 33, 65, 129, 193):
        for fp8 in (False, True):
            if fp8 and rows > 128:
                continue
            for n in (4096, 24576):
                us = [ops._C.few_rows_gemm_us(rows, n, k, fp8)
                      for k in range(2048, 16385, 2048)]
                assert us == sorted(us) and us[0] > 3
            us = [ops._C.few_rows_gemm_us(rows, n, 4096, fp8)
                  for n in (2048, 8192, 32768, 131072)]
            assert us == sorted(us)
