"""Rules of the work splits: fp8 projections of few rows (the GEMM's few-row tiles, the MFMA
few-row kernels, the VALU form), the row statistics of the bf16 softmax."""

import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.dispatch import launchers as LA

A = 1 << 20


@pytest.mark.parametrize("M,N,K,swiglu,want", [
    (1, 14336, 4096, True, False), (2, 14336, 4096, True, True), (64, 3072, 1024, True, True),
    (16, 1536, 2048, True, False), (16, 4096, 4096, False, False), (2, 4096, 14336, False, True),
    (17, 64, 64, False, True)])
def test_few_row_tiles_preferred(M, N, K, swiglu, want):
    assert LA.gemm_few_preferred(M, N, K, swiglu, "nt", True) is want
    assert not LA.gemm_few_preferred(M, N, K, swiglu, "nt", False)
    assert not LA.gemm_few_preferred(M, N, K, swiglu, "nn", True)


@pytest.mark.parametrize("M,suffix", [(1, "_kh32"), (32, "_kh32"), (33, "_kh64"), (64, "_kh64"), (65, "_kh"),
                                      (32768, "")])
def test_row_tiles_follow_the_rows(M, suffix):
    l = LA.gemm(A, A, A, M, 256, 256, layout="nt", b_dtype=dt.float8_e4m3fn, c_dtype=dt.bfloat16, scale_ptr=A,
                tile=128)
    assert l.symbol == "nk_gemm128_nt_e4m3_bf16" + suffix
    with pytest.raises(LA.LaunchError):
        LA.gemm(A, A, A, 65, 256, 256, layout="nt", b_dtype=dt.float8_e4m3fn, c_dtype=dt.bfloat16, scale_ptr=A,
                tile=128, kh=64)


@pytest.mark.parametrize("S,heads,want", [(24, 32, (4, 1, 1)), (649, 16, (4, 6, 21)), (1500, 32, (16, 3, 24)),
                                          (1800, 8, (8, 8, 64)), (5000, 4, (20, 8, 180)), (5000, None, (20, 8, 180))])
def test_row_statistics_chunks(S, heads, want):
    assert LA.attention_stat_chunks(S, True, heads) == want
    # whole query blocks of keys, so that no chunk starts past its queries
    assert want[0] % 4 == 0 and want[1] <= 8


@pytest.mark.parametrize("M,N,four", [(1 << 10, 1 << 7, True), (1 << 10, 127, False), ((1 << 15) - 1, 1 << 16, True),
                                      (1 << 15, 1 << 16, False), (1 << 16, (1 << 16) + 8, False)])
def test_reduction_of_large_outputs_keeps_64_bit_indices(M, N, four):
    """The form of four outputs per thread indexes rows and columns in 32
    bits: outputs of 2^31 elements and more take the other one."""
    out = LA.gemm_splitk(A, A, A, M, N, 128, layout="nt", b_dtype=dt.bfloat16, c_dtype=dt.bfloat16, ws_ptr=A,
                         split=(2, 64))[-1]
    assert out.symbol == "nk_gemv_out_bf16" and bool(out.args.flags & LA.GEMV_OUT4) is four
    assert out.grid[0] == -(-M * N // (1024 if four else 64))


@pytest.mark.parametrize("M,N,K,want", [(2, 4096, 4096, False), (32, 4096, 4096, False), (2, 3072, 2048, False),
                                        (16, 4096, 8192, False), (24, 4096, 8192, True), (4, 6144, 4096, False),
                                        (8, 12288, 4096, True), (2, 14336, 4096, True), (16, 6144, 2048, True),
                                        (8, 3072, 1024, True), (48, 4096, 4096, True)])
def test_few_row_tiles_of_a_pair_follow_the_models(M, N, K, want):
    """A SwiGLU pair whose K loop is long for its tiles, or runs in ranges,
    stays on the MFMA few-row kernels."""
    assert LA.gemm_few_preferred(M, N, K, True, "nt", True) is want
