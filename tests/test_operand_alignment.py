"""Operands that the fused kernels' 16-byte accesses cannot address: the
lowering leaves them to the kernels that take any address."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.core import tensor_apis
from nkipy_amd.core.trace import NKIPyKernel
from nkipy_amd.dispatch.launchers import LaunchError
from nkipy_amd.dispatch.lower import lower
from nkipy_amd.kernels import causal_gqa_attention_kernel
from nkipy_amd.kernels.qwen3 import apply_rotary_emb_kernel, compute_cos_sin_cache, prefill_attention_kernel
from nkipy_amd.kernels.rmsnorm import rmsnorm_kernel
from nkipy_amd.runtime import DeviceKernel, DeviceTensor
from nkipy_amd.runtime.device_tensor import DeviceBuffer

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


class _Shifted:
    """A buffer whose contents start 2 bytes after an allocation's."""

    def __init__(self, nbytes):
        self.base = DeviceBuffer(nbytes + 32)
        self.is_freed, self.ptr = False, self.base.ptr + 2

    def _live(self):
        self.base._live()

    def write(self, host, nbytes, offset=0):
        self.base.write(host, nbytes, offset + 2)

    def read(self, host, nbytes, offset=0):
        self.base.read(host, nbytes, offset + 2)


def _shifted(a, name):
    t = DeviceTensor(_Shifted(a.nbytes), a.shape, a.dtype, name)
    t.write_from_numpy(a)
    return t


def _attention(xq, xk, xv):
    return causal_gqa_attention_kernel(xq, xk, xv)


def _cached(qkv, q_weight, k_weight, cache_k, cache_v):
    xq = _prefill(0)(qkv, q_weight, k_weight, cache_k, cache_v)
    return prefill_attention_kernel(xq, cache_k, cache_v)


@pytest.mark.gpu
@pytest.mark.parametrize("fn,shifted", [(_attention, {"xq", "xk", "xv", "output0"}), (_attention, {"xk"}),
                                        (_cached, {"cache_k", "cache_v"}), (_cached, {"cache_v", "output0"})])
def test_ragged_attention_at_any_address(gpu, fn, shifted):
    """Arguments between 16-byte boundaries, which the unfused kernels of such
    lengths take: the aligned call's results, caches updated in place, for the
    values of each call; and through a graph."""
    B, S = 2, 35
    print(f"shifted {fn.__name__} {sorted(shifted)}", flush=True)
    rng = np.random.default_rng(S)
    shapes = [(B, S, n, D) for n in (H, HKV, HKV)] if fn is _attention else \
        [(B, S, (H + 2 * HKV) * D), (D,), (D,), (B, 48, HKV, D), (B, 48, HKV, D)]
    draw = lambda: [dt.to_bf16(rng.standard_normal(s).astype(np.float32)) for s in shapes]
    args = draw()
    dk = DeviceKernel.compile_and_load(fn, *args, name=f"shifted_{fn.__name__}")
    names = [n.split(".must_alias_input")[0] for n in dk.input_tensors_info]
    sets = []
    for move in (set(), shifted):
        put = lambda n, a: _shifted(a, n) if n in move else DeviceTensor.from_numpy(a, name=n)
        ins = {full: put(n, a) for full, n, a in zip(dk.input_tensors_info, names, args)}
        outs = {n: ins[f"{n}.must_alias_input"] if n in names else
                put(n, np.zeros(i.shape, dt.canonical(i.dtype))) for n, i in dk.output_tensors_info.items()}
        sets.append((ins, outs))
    for graph in (False, False, True):
        got = []
        for ins, outs in sets:
            for t, a in zip(ins.values(), args):
                t.write_from_numpy(a)
            dk(ins, outs, graph=graph)
            got.append({n: dt.numpy_storage(t.numpy()).tobytes() for n, t in outs.items()})
        assert got[0] == got[1]
        args = draw()


@pytest.mark.gpu
def test_whole_blocks_still_want_alignment(gpu):
    z = [np.zeros((1, 128, n, D), dt.bfloat16) for n in (H, HKV, HKV)]
    dk = DeviceKernel.compile_and_load(_attention, *z, name="shifted_whole")
    ins = {n: _shifted(a, n) for n, a in zip(dk.input_tensors_info, z)}
    with pytest.raises(LaunchError):
        dk(ins)
