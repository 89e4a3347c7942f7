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
