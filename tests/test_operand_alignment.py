"""Operands that the fused kernels' 16-byte accesses cannot address: the
lowering leaves them to the kernels that take any address."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.core import tensor_apis
from nkipy_amd.core.trace import NKIPyKernel
from nkipy_amd.dispatch.lower import lower
from nkipy_amd.kernels.qwen3 import apply_rotary_emb_kernel, compute_cos_sin_cache
from nkipy_amd.kernels.rmsnorm import rmsnorm_kernel

H, HKV, D = 4, 2, 128


def _prefill(gap):
    """A prefill prologue whose v heads start ``gap`` columns after k's."""
    def fn(qkv, q_weight, k_weight, cache_k, cache_v):
        B, S, _ = qkv.shape
        v0 = (H + HKV) * D + gap
        xq = rmsnorm_kernel(qkv[:, :, :H * D].reshape(B, S, H, D), q_weight, 1e-6)
        xk = rmsnorm_kernel(qkv[:, :, H * D:(H + HKV) * D].reshape(B, S, HKV, D), k_weight, 1e-6)
        cos, sin = compute_cos_sin_cache(D, cache_k.shape[1], base=1.0e6)
        cos = tensor_apis.constant(cos).astype(qkv.dtype)[:S]
        sin = tensor_apis.constant(sin).astype(qkv.dtype)[:S]
        xq, xk = apply_rotary_emb_kernel(xq, xk, cos, sin)
        cache_k[:, :S] = xk
        cache_v[:, :S] = qkv[:, :, v0:v0 + HKV * D].reshape(B, S, HKV, D)
        return xq
    return fn


@pytest.mark.parametrize("gap,kinds", [(0, ["head_rope"]), (8, ["head_rope"]), (4, None), (1, None)])
def test_prologue_copies_only_aligned_heads(gap, kinds):
    """The prologue's launch writes the caches where the v heads lie in whole
    16-byte pieces of the projection; elsewhere programs do."""
    z = lambda *s: np.zeros(s, dt.bfloat16)
    plan = lower(NKIPyKernel.trace(_prefill(gap)).specialize(
        z(2, 5, (H + 2 * HKV) * D + 8), z(D), z(D), z(2, 16, HKV, D), z(2, 16, HKV, D)))
    symbols = [l.symbol for st in plan.steps for l in st.launches(lambda v: 1 << 40)]
    assert "nk_head_rope_bf16" in symbols
    assert plan.kernel_kinds == kinds if kinds else "elementwise" in plan.kernel_kinds
