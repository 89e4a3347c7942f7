"""Softmax of rows that are not in whole 16-byte pieces: every register form's
edges and the loop past them, against float64."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.dispatch import launchers as LA
from nkipy_amd.runtime import DeviceTensor

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
