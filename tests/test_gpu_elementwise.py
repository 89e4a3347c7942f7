"""The float form of the elementwise programs (nk_ew_f32) against the general
kernel (nk_ew_program), bit for bit: every operation it takes, result types,
broadcast, transposed, sliced and odd-sized operands, special values; and the
host's collapsing of dimensions on the CPU."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.core.trace import NKIPyKernel
from nkipy_amd.dispatch import generic as G
from nkipy_amd.dispatch.lower import lower
from nkipy_amd.runtime import DeviceKernel, DeviceTensor


def _unary(x, y):
    outs = [np.exp(x), np.log(np.abs(x)), np.sqrt(np.abs(x)), np.tanh(x), np.ceil(x), np.floor(x), np.rint(x),
            np.trunc(x), np.sign(x), -x, 1 / (1 + np.exp(-y))]
    acc = outs[0]
    for o in outs[1:]:
        acc = np.where(acc > o, acc * 0.5, acc - o)
    return acc, np.logical_not(np.isfinite(x)), np.isnan(y)


def _binary(x, y):
    a = (x + y) * (x - y)
    b = np.maximum(a, x) / np.minimum(y, a)
    return a, b, np.where(np.less_equal(x, y), a, b), np.equal(x, y), np.greater_equal(x, b)


def _views(x, y):
    t = np.transpose(x) * 2.0 if x.ndim == 2 else x * 2.0
    row = np.expand_dims(x[..., 0], -1) + y
    return t, row, x[..., 1:] - y[..., :-1], np.broadcast_to(y[:1], y.shape) * x


def _casts(x, y):
    h = x.astype(np.float16) * y.astype(np.float16)
    return h, h.astype(np.float32) + x, (x > y).astype(np.float32)


PROGRAMS = {"unary": _unary, "binary": _binary, "views": _views, "casts": _casts}


def _both(fn, args, monkeypatch):
    g = NKIPyKernel.trace(fn).specialize(*args)
    names = [p.name for p in g.parameters]
    res, symbols = [], []
    for i, general in enumerate((False, True)):
        if general:
            monkeypatch.setattr(G.ProgramStep, "_float_form", lambda self, addr, total: None)
        plan = lower(g)
        dk = DeviceKernel(g, plan, f"elementwise_{i}")
        out = dk({n: DeviceTensor.from_numpy(a, name=n) for n, a in zip(names, args)})
        res.append({k: v.numpy().tobytes() for k, v in out.items()})
        symbols.append({l.symbol for st in plan.steps for l in st.launches(lambda v: 1 << 40)})
    return res, symbols


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(PROGRAMS))
@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (64, 64), (37, 260), (130, 1001), (2, 3, 8)])
@pytest.mark.parametrize("d", ["float32", "float16", "bfloat16"])
def test_float_form_equals_the_general_kernel(gpu, monkeypatch, name, shape, d):
    if name == "casts" and d == "bfloat16":
        pytest.skip("bf16 arrays have no NumPy fp16 cast without ml_dtypes")
    print(f"elementwise {name} {shape} {d}", flush=True)
    rng = np.random.default_rng(len(name) + shape[-1])
    arrays = []
    for _ in range(2):
        a = (rng.standard_normal(shape) * 4).astype(np.float32)
        flat = a.reshape(-1)
        special = [0.0, -0.0, np.inf, -np.inf, np.nan, 1e-41, -3e-42, 88.8, -104.0, 0.5, 2.5]
        pick = rng.integers(0, flat.size, min(flat.size, len(special)))
        flat[pick] = special[:len(pick)]
        arrays.append(dt.to_bf16(a) if d == "bfloat16" else a.astype(d))
    res, symbols = _both(PROGRAMS[name], arrays, monkeypatch)
    assert "nk_ew_f32" in symbols[0] and "nk_ew_f32" not in symbols[1]
    for k in res[0]:
        assert res[0][k] == res[1][k], k


def test_collapse_dims():
    full = lambda sh: list(G.contiguous_strides(sh))
    assert G.collapse_dims((2, 3, 4), [full((2, 3, 4))] * 2) == ([24], [[1], [1]])
    # a broadcast row: the outer two merge, the row stays
    assert G.collapse_dims((2, 3, 4), [full((2, 3, 4)), [0, 0, 1]]) == ([6, 4], [[4, 1], [0, 1]])
    # a transpose merges nothing; size-1 dimensions go
    assert G.collapse_dims((3, 1, 4), [full((3, 1, 4)), [1, 7, 3]]) == ([3, 4], [[4, 1], [1, 3]])
    assert G.collapse_dims((1, 1), [[1, 1]]) == ([1], [[0]])


def _ragged(x, y, z):
    t = np.transpose(y)
    m = np.greater(x, t)
    return x + t * z, np.where(m, np.flip(x, axis=0), z), m, np.flip(t, axis=x.ndim - 1) - x


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(5, 3, 2), (7, 1, 3), (2, 3, 2, 3, 3), (3, 2, 2, 3, 2, 3), (9, 5), (130, 1001)])
@pytest.mark.parametrize("d", ["float32", "float16", "bfloat16"])
def test_ragged_rows_equal_the_general_kernel(gpu, monkeypatch, shape, d):
    """Innermost dimensions shorter than, or no multiple of, a thread's four
    elements, at the sizes that the rule leaves to the general kernel too:
    reversed, transposed and broadcast operands, a mask."""
    print(f"elementwise ragged {shape} {d}", flush=True)
    monkeypatch.setattr(G, "EWF_RAGGED_MIN", -1)
    rng = np.random.default_rng(len(shape))
    arrays = [rng.standard_normal(s).astype(np.float32) for s in (shape, shape[::-1], shape[-1:])]
    res, symbols = _both(_ragged, [dt.to_bf16(x) if d == "bfloat16" else x.astype(d) for x in arrays], monkeypatch)
    assert symbols[0] == {"nk_ew_f32"} and "nk_ew_f32" not in symbols[1]
    assert res[0] == res[1]


@pytest.mark.gpu
@pytest.mark.parametrize("d", ["float16", "bfloat16"])
def test_functions_of_every_16_bit_value(gpu, monkeypatch, d):
    """The functions evaluated in double reach their 16-bit type in one
    rounding: by way of fp32 about ten fp16 results (exp(0.02269), just below
    the middle of two) fall on a tie that the true value is not on."""
    print(f"elementwise functions {d}", flush=True)
    bits = np.arange(65536, dtype=np.uint16).reshape(64, 1024)
    x = dt.to_bf16((bits.astype(np.uint32) << 16).view(np.float32)) if d == "bfloat16" else bits.view(np.float16)

    def fn(x):
        return np.exp(x), np.log(x), np.sqrt(x), np.tanh(x), 1 / (1 + np.exp(-x))

    res, symbols = _both(fn, [x], monkeypatch)
    # a program a result: the roots (no function) stay on the plain kernel
    assert "nk_ew_f32" in symbols[0] and ("nk_ew_f32_f16fn" in symbols[0]) == (d == "float16")
    assert "nk_ew_program" not in symbols[0] and symbols[1] == {"nk_ew_program"}

    def values(raw):
        raw = np.frombuffer(raw, np.uint16).reshape(x.shape)
        return (raw.astype(np.uint32) << 16).view(np.float32) if d == "bfloat16" else raw.view(np.float16)

    for k in res[0]:
        np.testing.assert_array_equal(values(res[0][k]), values(res[1][k]), err_msg=k)
    if d == "float16":
        with np.errstate(all="ignore"):
            for k, f in zip(res[0], (np.exp, np.log, np.sqrt, np.tanh)):
                want = f(bits.view(np.float16).astype(np.float64)).astype(np.float16)
                np.testing.assert_array_equal(values(res[0][k]), want, err_msg=k)


@pytest.mark.parametrize("shape,symbol", [((1000, 33), "nk_ew_program"), ((1000, 32), "nk_ew_f32"),
                                          ((3971, 33), "nk_ew_program"), ((3972, 33), "nk_ew_f32"),
                                          ((1, 33), "nk_ew_f32")])
def test_small_ragged_programs_take_the_general_kernel(shape, symbol):
    x, row = np.zeros(shape, np.float32), np.zeros(shape[-1:], np.float32)
    plan = lower(NKIPyKernel.trace(lambda x, y: x + y).specialize(x, row))
    assert [l.symbol for st in plan.steps for l in st.launches(lambda v: 1 << 40)] == [symbol]
