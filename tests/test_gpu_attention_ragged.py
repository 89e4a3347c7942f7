"""Attention over sequence lengths that are no multiple of the 128-query
block, on the GPU: the fp32-softmax form against the float64 oracle and the
bf16-softmax form against the op-by-op oracle, at the lengths around the
edges of a wave's 32 queries, a 32-key block, a query block and the row
statistics' 512-key chunks, masked and unmasked."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.core.trace import NKIPyKernel
from nkipy_amd.dispatch.lower import lower
from nkipy_amd.kernels import causal_gqa_attention_kernel
from nkipy_amd.kernels.qwen3 import prefill_attention_kernel
from nkipy_amd.kernels.softmax import softmax_kernel
from nkipy_amd.runtime import DeviceKernel, DeviceTensor
from oracle import kernels as K
from oracle import numerics as N

LENGTHS = [2, 8, 31, 33, 127, 129, 200, 353, 513, 1000]
D = 128


def _unmasked(xq, xk, xv):
    rep = xq.shape[2] // xk.shape[2]
    q = xq.transpose(0, 2, 1, 3).astype(np.float32)
    kt = np.repeat(xk, rep, axis=2).transpose(0, 2, 3, 1).astype(np.float32)
    v = np.repeat(xv, rep, axis=2).transpose(0, 2, 1, 3).astype(np.float32)
    p = softmax_kernel(np.matmul(q, kt) / np.float32(np.sqrt(D)))
    return np.matmul(p, v).transpose(0, 2, 1, 3).astype(xq.dtype)


def _unmasked_bf16(xq, xk, xv):
    rep = xq.shape[2] // xk.shape[2]
    q = xq.transpose(0, 2, 1, 3)
    k = np.repeat(xk, rep, axis=2).transpose(0, 2, 1, 3)
    v = np.repeat(xv, rep, axis=2).transpose(0, 2, 1, 3)
    s = ((q @ k.transpose(0, 1, 3, 2)) / np.float32(np.sqrt(D))).astype(xq.dtype)
    return (softmax_kernel(s) @ v).transpose(0, 2, 1, 3)


def _qkv(B, S, Hq, Hkv, keys=None):
    rng = np.random.default_rng(S + Hq)
    return [N.bf16_round(rng.standard_normal((B, n, h, D)))
            for n, h in ((S, Hq), (keys or S, Hkv), (keys or S, Hkv))]


def _call(fn, arrays, name):
    args = [dt.to_bf16(a) for a in arrays]
    dk = DeviceKernel.compile_and_load(fn, *args, name=name)
    assert dk.plan.kernel_kinds == ["attention"], dk.plan.kernel_kinds
    ins = {n: DeviceTensor.from_numpy(a, name=n) for n, a in zip(dk.input_tensors_info, args)}
    return dt.to_float32(dk(ins)["output0"].numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("S", LENGTHS)
def test_fp32_softmax(gpu, S, causal):
    B, Hq, Hkv = 2, 4, 2
    print(f"ragged attention S={S} causal={causal}", flush=True)
    q, k, v = _qkv(B, S, Hq, Hkv)
    got = _call(causal_gqa_attention_kernel if causal else _unmasked, (q, k, v), f"rag_{S}_{causal}")
    q, k, v = (np.asarray(a, np.float64).transpose(0, 2, 1, 3) for a in (q, k, v))
    k, v = (np.repeat(a, Hq // Hkv, axis=1) for a in (k, v))
    s = q @ k.transpose(0, 1, 3, 2) / np.sqrt(D)
    if causal:
        s = np.where(np.triu(np.ones((S, S), bool), 1), -np.inf, s)
    w = np.exp(s - s.max(-1, keepdims=True))
    ref = (w / w.sum(-1, keepdims=True) @ v).transpose(0, 2, 1, 3)
    got = got.reshape(ref.shape)
    # one bf16 rounding of the result (8 significant bits: at most 2^-8 of the
    # value), plus weights good to 2^-17 and fp32 sums, which the largest
    # value bounds
    bound = 2.0 ** -8 * np.abs(ref) + 2.0 ** -15 * np.abs(v).max()
    worst = float(np.max(np.abs(got - ref) / bound))
    assert worst <= 1.0


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("S", LENGTHS)
def test_bf16_softmax(gpu, S, causal):
    B, Hq, Hkv = 2, 4, 2
    print(f"ragged bf16 attention S={S} causal={causal}", flush=True)
    q, k, v = _qkv(B, S, Hq, Hkv, keys=1152 if causal else None)
    got = _call(prefill_attention_kernel if causal else _unmasked_bf16, (q, k, v), f"ragb_{S}_{causal}")
    ref = K.qwen3_prefill_attention(q, k, v, rows=np.arange(S), causal=causal)
    # every cast point is the traced code's: the order of the fp32 sums moves
    # a rounding across a bf16 boundary now and then
    same = float(np.mean(got == ref))
    rms = np.sqrt(np.mean(ref ** 2, axis=-1, keepdims=True))
    worst = float(np.max(np.abs(got - ref) / (2e-2 * np.abs(ref) + 2e-2 * rms)))
    print(f"identical {same:.5f}, worst {worst:.3f} of the bar", flush=True)
    assert same >= 0.995 and worst <= 1.0


@pytest.mark.parametrize("S", [2, 200, 384])
def test_lowering_takes_every_length(S):
    """Both traced forms lower to the attention step at any length; the
    ragged kernels are taken exactly where the query blocks are partial."""
    z = np.zeros((2, S, 4, D), dt.bfloat16), np.zeros((2, S, 2, D), dt.bfloat16)
    plan = lower(NKIPyKernel.trace(causal_gqa_attention_kernel).specialize(z[0], z[1], z[1]))
    cache = np.zeros((2, 512, 2, D), dt.bfloat16)
    bplan = lower(NKIPyKernel.trace(prefill_attention_kernel).specialize(z[0], cache, cache))
    assert plan.kernel_kinds == bplan.kernel_kinds == ["attention"]
    symbols = [l.symbol for p in (plan, bplan) for st in p.steps for l in st.launches(lambda v: 1 << 40)
               if "causal" in l.symbol]
    assert [("_rag" in s) for s in symbols] == [S % 128 != 0] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("S", [35, 129, 353])
def test_weights_keep_fp32(gpu, S):
    """The weights of the fp32 softmax enter P V as fp32: value columns that
    subtract a weight's leading 16 bits leave its last ones, which the bf16
    output then shows.  Query 0's scores are 0 for three keys (p = 1) and -t
    for a fourth; v sums to p - hi - mid with hi, mid the leading two groups
    of eight bits of p = exp(-t)."""
    rng = np.random.default_rng(S)
    t = N.bf16_round(rng.uniform(0.05, 3, D)).astype(np.float64)
    q = np.zeros((1, S, D, D))
    k, v = np.zeros((1, S, 1, D)), np.zeros((1, S, 1, D))
    keys = rng.permutation(S)[:4]
    other = np.setdiff1d(np.arange(S), keys)
    q[0, :, :, 0] = 2.0 ** 10  # every other key: a score of -2^15, weight 0
    k[0, other, 0, 0] = -2.0 ** 5 * np.sqrt(D).astype(np.float32)
    # head h: scores of the fourth key -t[h]
    q[0, :, :, 1] = -t
    k[0, keys[3], 0, 1] = 1.0
    p = np.exp(-t / np.sqrt(D))
    hi = N.bf16_round(p).astype(np.float64)
    mid = N.bf16_round(p - hi).astype(np.float64)
    # one column of v per head: the head's own column is read back
    v[0, keys[0], 0], v[0, keys[1], 0], v[0, keys[3], 0] = -hi, -mid, 1.0
    args = [N.bf16_round(a) for a in (q, k, v)]
    assert np.array_equal(args[2], v)
    got = _call(_unmasked, args, f"rag_weights_{S}").reshape(S, D, D)
    left = np.array([got[:, h, h] for h in range(D)], np.float64) * (3 + p)[:, None]
    # 2^-21 of the weight: its exponent's argument, the hardware's 2^x (1 ulp)
    # and the fp32 sums, about 2^-24 each; the value subtracted to is at most
    # 2^-18 of it, bf16 there is exact to 2^-26
    worst = float(np.max(np.abs(left - (p - hi - mid)[:, None]) / p[:, None]))
    print(f"weights to 2^{np.log2(worst):.1f}, left {np.max(np.abs(p - hi - mid)):.2e}", flush=True)
    assert worst <= 2.0 ** -21


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
def test_infinite_values(gpu, causal):
    """An infinite v comes out infinite in every query that sees its key, in
    its column alone."""
    S, at = 200, 70
    q, k, v = _qkv(1, S, 2, 1)
    v[0, at, 0, 5], v[0, at, 0, 9] = np.inf, -np.inf
    got = _call(causal_gqa_attention_kernel if causal else _unmasked, (q, k, v), f"rag_inf_{causal}")
    sees = got.reshape(1, S, 2, D)[0, at if causal else 0:]
    assert np.all(sees[..., 5] == np.inf) and np.all(sees[..., 9] == -np.inf)
    assert np.all(np.isfinite(np.delete(sees, [5, 9], axis=-1)))
