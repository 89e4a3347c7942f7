"""Softmax of rows that are not in whole 16-byte pieces: every register form's
edges and the loop past them, against float64."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.dispatch import launchers as LA
from nkipy_amd.runtime import DeviceTensor
from oracle import numerics as N

LENGTHS = [1, 63, 65, 250, 257, 1023, 1025, 2047, 2049, 4095, 4097, 8191, 8193, 16383, 16385, 32767, 32769]


def test_forms_by_length():
    sym = lambda n, **kw: LA.softmax_rows(1 << 20, 1 << 20, 4, n, dt.float32, dt.float32, **kw).symbol
    assert sym(255) == "nk_softmax_elt_f32_f32_b64_e4" and sym(257) == "nk_softmax_elt_f32_f32_b256_e4"
    assert sym(32767) == "nk_softmax_elt_f32_f32_b512_e64" and sym(32769) == "nk_softmax_loop_f32_f32"
    assert sym(256).startswith("nk_softmax_reg")


@pytest.mark.gpu
@pytest.mark.parametrize("ti,to", sorted(LA._SOFTMAX_TYPES))
@pytest.mark.parametrize("n", LENGTHS)
def test_ragged_rows(gpu, n, ti, to):
    types = {"f32": dt.float32, "bf16": dt.bfloat16, "f16": dt.float16}
    print(f"softmax {n} {ti}->{to}", flush=True)
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((3, n)) * 4).astype(np.float32)
    x[1, : n // 2] = -np.inf
    x[2] = -3e4  # equal weights
    host = dt.to_bf16(x) if ti == "bf16" else x.astype(types[ti])
    x = dt.to_float32(host) if ti == "bf16" else host.astype(np.float32)
    src, out = DeviceTensor.from_numpy(host), DeviceTensor.empty((3, n), types[to])
    LA.softmax_rows(src.ptr, out.ptr, 3, n, types[ti], types[to]).run(gpu)
    gpu.sync()
    got = dt.to_float32(out.numpy()) if to == "bf16" else out.numpy().astype(np.float32)
    e = np.exp(x.astype(np.float64) - x.max(-1, keepdims=True))
    ref = e / e.sum(-1, keepdims=True)
    # fp32 exponentials, sums of n terms and one quotient, then the output's
    # rounding (fp16: its subnormal step below 2^-14)
    last = {"f32": 2.0 ** -22, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}[to]
    bound = ref * (last + 2.0 ** -20 + np.sqrt(n) * 2.0 ** -23) + (2.0 ** -24 if to == "f16" else 1e-37)
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("ti,to", sorted(LA._SOFTMAX_TYPES))
@pytest.mark.parametrize("n", [1, 63, 257, 1025, 4097, 8193, 16385, 32769])
def test_rows_without_a_finite_maximum(gpu, n, ti, to):
    """A NaN anywhere, a row of -inf alone and a +inf make their whole row
    NaN, as x - max and the sum do; the rows beside them stay as they are."""
    types = {"f32": dt.float32, "bf16": dt.bfloat16, "f16": dt.float16}
    print(f"softmax special {n} {ti}->{to}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((6, n)).astype(np.float32)
    x[1, n // 2], x[2], x[3, n - 1], x[4, 0] = np.nan, -np.inf, np.inf, np.nan
    cast = lambda a: dt.to_bf16(a) if ti == "bf16" else a.astype(types[ti])
    widen = lambda t: dt.to_float32(t.numpy()) if to == "bf16" else t.numpy().astype(np.float32)
    outs = []
    for a in (x, x[[0, 5]]):
        src, out = DeviceTensor.from_numpy(cast(a)), DeviceTensor.empty(a.shape, types[to])
        LA.softmax_rows(src.ptr, out.ptr, len(a), n, types[ti], types[to]).run(gpu)
        gpu.sync()
        outs.append(widen(out))
    assert np.all(np.isnan(outs[0][1:5]))
    np.testing.assert_array_equal(outs[0][[0, 5]], outs[1])
    assert np.all(np.isfinite(outs[1]))


@pytest.mark.gpu
@pytest.mark.parametrize("d", ["bf16", "f16"])
@pytest.mark.parametrize("n", LENGTHS)
def test_rounded_steps(gpu, n, d):
    """The softmax whose steps round to its 16-bit type, at every form's edges:
    against the same steps on float64 values rounded to that type."""
    print(f"softmax rounded {n} {d}", flush=True)
    ty, bits = (dt.bfloat16, 8) if d == "bf16" else (dt.float16, 11)
    rnd = N.bf16_round if d == "bf16" else (lambda a: a.astype(np.float16))
    rng = np.random.default_rng(n)
    x = np.asarray(rnd((rng.standard_normal((3, n)) * 2).astype(np.float32)), np.float32)
    x[1, : n // 2] = -np.inf
    src = DeviceTensor.from_numpy(dt.to_bf16(x) if d == "bf16" else x.astype(np.float16))
    out = DeviceTensor.empty((3, n), ty)
    LA.softmax_rows(src.ptr, out.ptr, 3, n, ty, ty, round_ops=True).run(gpu)
    gpu.sync()
    got = dt.to_float32(out.numpy()) if d == "bf16" else out.numpy().astype(np.float32)
    r = lambda a: np.asarray(rnd(np.asarray(a, np.float32)), np.float64)
    e = r(np.exp(r(x - x.max(-1, keepdims=True))))
    s = e.sum(-1, keepdims=True)
    ref = e / r(s)
    # the result's rounding, and a step of e or of the sum that falls the other
    # way (2^-bits each at most); fp16: its subnormal step
    bound = ref * 4 * 2.0 ** -bits + (2.0 ** -23 if d == "f16" else 1e-37)
    assert np.all(np.abs(got - ref) <= bound)
