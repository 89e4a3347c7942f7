"""The rule that picks a GEMM's output tile and K ranges (gemm_form)."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.core.trace import NKIPyKernel
from nkipy_amd.dispatch import launchers as LA
from nkipy_amd.dispatch.lower import lower

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


@pytest.mark.parametrize("layout,fp8", [("nt", True), ("nt", False), ("nn", False), ("nn", True)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_every_form_is_one_the_launchers_take(layout, fp8, swiglu):
    """Over rows, widths and depths in use and odd ones: the ranges cover K,
    the planes stay within their bound, and the launchers build the form."""
    kw = dict(layout=layout, b_dtype=dt.float8_e4m3fn if fp8 else dt.bfloat16, c_dtype=dt.bfloat16,
              scale_ptr=A if fp8 else 0)
    if swiglu:
        kw.update(up_ptr=A, up_scale_ptr=A if fp8 else 0)
    for M in (1, 2, 17, 32, 33, 64, 65, 100, 128, 129, 300, 513, 1000, 2049, 4096, 8192, 8193, 10000):
        for N, K in ((64, 64), (72, 80), (520, 1056), (1536, 2048), (2048, 1536), (3072, 1024), (4096, 4096),
                     (6144, 4096), (14336, 4096), (4096, 14336), (151936, 1024)):
            tile, ks, kc = LA.gemm_form(M, N, K, layout, fp8, swiglu)
            assert tile in (64, 128, 256)
            if ks > 1:
                assert tile == 128 and kc % 64 == 0 and ks == -(-K // kc) and ks <= LA.GEMM128_MAX_RANGES
                assert 4 * ks * M * N * (2 if swiglu else 1) <= 1 << 28
                ls = LA.gemm_splitk(A, A, A, M, N, K, ws_ptr=A, split=(ks, kc), **kw)
                assert [l.grid[1] for l in ls[:-1]] == [ks] * (2 if swiglu else 1)
            else:
                l = LA.gemm(A, A, A, M, N, K, tile=tile, **kw)
                assert l.grid[0] == -(-M // tile) * -(-N // (max(tile, 128) // (2 if swiglu else 1)))
            assert LA.gemm_form(M, N, K, layout, fp8, swiglu, False)[1] == 1


def _nn(x, w):
    return np.matmul(x, w)


def _nt8(x, w, s):
    return np.matmul(x, np.transpose((w.astype(np.float32) * np.expand_dims(s, 1)).astype(x.dtype)))


@pytest.mark.parametrize("fn,M,N,K,symbols", [
    (_nt8, 170, 6144, 4096, ["nk_gemm128_nt_e4m3_bf16_kh64"]),
    (_nt8, 1000, 4096, 4096, ["nk_gemm128_nt_e4m3_bf16_kh"]),
    (_nt8, 2000, 4096, 4096, ["nk_gemm128_nt_e4m3_bf16"]),
    (_nn, 4096, 12288, 4096, ["nk_gemm8k_nn_bf16_bf16_r16"]),
    (_nn, 300, 4096, 12288, ["nk_gemm128_nn_bf16_f32_splitk", "nk_gemv_out_bf16"]),
    (_nt8, 24, 4096, 14336, ["nk_gemm8k_nt_e4m3_f32_splitk32", "nk_gemv_out_bf16"])])
def test_lowered_projections(fn, M, N, K, symbols):
    x = np.zeros((M, K), dt.bfloat16)
    w = [np.zeros((K, N), dt.bfloat16)] if fn is _nn else [np.zeros((N, K), dt.float8_e4m3fn), np.zeros(N, np.float32)]
    plan = lower(NKIPyKernel.trace(fn).specialize(x, *w))
    assert [l.symbol for st in plan.steps for l in st.launches(lambda v: 1 << 40)] == symbols
