"""SwiGLU over a fp32 product's partial planes (nk_swiglu_planes_f32): the same
bits as the planes' reduction and the elementwise program, and when the
lowering takes it."""

import numpy as np
import pytest

from nkipy_amd.core.trace import NKIPyKernel
from nkipy_amd.dispatch import generic as G
from nkipy_amd.dispatch.lower import lower
from nkipy_amd.kernels import feedforward_kernel
from nkipy_amd.runtime import DeviceKernel, DeviceTensor, baremetal_jit


def _half(x, w):
    g, u = np.split(np.matmul(x, w), 2, axis=-1)
    return g * (1 / (1 + np.exp(-g))) * u


def _swapped(x, w):
    u, g = np.split(np.matmul(x, w), 2, axis=-1)
    return u * ((1 / (np.exp(-g) + 1)) * g)


def _plan(fn, *shapes, dtype=np.float32):
    return lower(NKIPyKernel.trace(fn).specialize(*[np.zeros(s, dtype) for s in shapes]))


def test_taken_for_the_product_alone():
    assert _plan(feedforward_kernel, (20, 64), (64, 256), (128, 64)).kernel_kinds == ["dot", "swiglu", "dot"]
    st = _plan(_swapped, (2, 3, 64), (64, 256)).steps[1]
    assert st.kind == "swiglu" and st.cols == (128, 0)

    def kept(x, w):
        y = np.matmul(x, w)
        g, u = np.split(y, 2, axis=-1)
        return g * (1 / (1 + np.exp(-g))) * u, y

    def silu_of_both(x, w):
        g, u = np.split(np.matmul(x, w), 2, axis=-1)
        return g * (1 / (1 + np.exp(-u))) * u

    def other_constant(x, w):
        g, u = np.split(np.matmul(x, w), 2, axis=-1)
        return g * (1 / (2 + np.exp(-g))) * u

    for fn in (kept, silu_of_both, other_constant):
        assert "swiglu" not in _plan(fn, (20, 64), (64, 256)).kernel_kinds
    # columns that take no vectors of four; half-precision products
    assert "swiglu" not in _plan(_half, (20, 64), (64, 254)).kernel_kinds
    assert "swiglu" not in _plan(_half, (20, 64), (64, 256), dtype=np.float16).kernel_kinds


@pytest.mark.gpu
@pytest.mark.parametrize("fn", [_half, _swapped])
@pytest.mark.parametrize("lead,K,F", [((1,), 32, 4), ((2,), 2048, 132), ((2, 3), 700, 64), ((65,), 96, 1000),
                                      ((300,), 256, 2048)])
def test_bits_of_the_two_launches(gpu, monkeypatch, fn, lead, K, F):
    print(f"swiglu planes {lead} {K} {F}", flush=True)
    rng = np.random.default_rng(K + F)
    x = rng.standard_normal(lead + (K,)).astype(np.float32)
    w = (rng.standard_normal((K, 2 * F)) * 4 / np.sqrt(K)).astype(np.float32)
    w[:, 1] *= 40.0  # gates whose exp overflows and underflows
    w[:, F + 1] = 0.0
    x[..., 0, 0] = 0.0
    got = np.asarray(baremetal_jit(fn)(x, w))
    assert "swiglu" in _plan(fn, x.shape, w.shape).kernel_kinds
    monkeypatch.setattr(G, "fuse_swiglu_planes", lambda plan: None)

    def plain(x, w):
        return fn(x, w)

    dk = DeviceKernel.compile_and_load(plain, x, w, name=f"plain_{fn.__name__}_{K}_{F}", use_cached_if_exists=False)
    assert "swiglu" not in dk.plan.kernel_kinds
    out = DeviceTensor.empty(got.shape, np.float32, name="output0")
    dk({"x": DeviceTensor.from_numpy(x, name="x"), "w": DeviceTensor.from_numpy(w, name="w")}, {"output0": out})
    assert np.array_equal(got.view(np.uint32), out.numpy().view(np.uint32))
