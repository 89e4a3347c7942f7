"""The rule that picks a GEMM's output tile and K ranges (gemm_form)."""

import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.dispatch import launchers as LA

A = 1 << 20


@pytest.mark.parametrize("layout,fp8", [("nt", True), ("nt", False), ("nn", False)])
@pytest.mark.parametrize("M,N,K", [(2, 64, 64), (17, 128, 128), (33, 256, 256), (64, 2048, 256)])
def test_few_rows_of_small_weights_take_the_few_row_tiles(M, N, K, layout, fp8):
    assert LA.gemm_form(M, N, K, layout, fp8)[0] == 128
    assert LA.gemm_form(M, N, K, layout, fp8, True)[0] == 128


@pytest.mark.parametrize("M,N,K,layout,fp8,swiglu,tile", [
    (198, 14336, 4096, "nn", False, True, 256), (591, 14336, 4096, "nt", False, True, 256),
    (1237, 7168, 5120, "nt", False, True, 256), (1269, 3072, 2048, "nn", False, True, 128),
    (214, 12288, 4096, "nt", False, True, 128), (165, 12288, 4096, "nt", True, True, 128),
    (2049, 4096, 14336, "nt", False, False, 256), (1757, 5120, 15360, "nt", True, False, 256),
    (1000, 4096, 4096, "nt", True, False, 128), (300, 4096, 12288, "nn", False, False, 128),
    (170, 6144, 4096, "nt", True, False, 64), (4096, 12288, 4096, "nn", False, False, 256)])
def test_small_tiles_only_where_they_gain(M, N, K, layout, fp8, swiglu, tile):
    """The 256 x 256 tiles where the smaller ones measured slower or tie."""
    assert LA.gemm_form(M, N, K, layout, fp8, swiglu)[0] == tile
