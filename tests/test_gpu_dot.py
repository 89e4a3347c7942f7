"""The strided fp32 product on the matrix cores (nk_dot_f32): every load
mode (contiguous along k, along rows / columns, neither), types, batches,
sizes around the tile, stage and range edges, traced from NumPy against
float64; the host rules on the CPU."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.core.trace import NKIPyKernel
from nkipy_amd.dispatch import generic as G
from nkipy_amd.dispatch.lower import lower
from nkipy_amd.runtime import DeviceKernel, DeviceTensor, baremetal_jit


def _nn(a, b):
    return np.matmul(a, b)


def _tn(a, b):
    return np.matmul(np.swapaxes(a, -1, -2), b)


def _nt(a, b):
    return np.matmul(a, np.swapaxes(b, -1, -2))


def _every_other(a, b):
    return np.matmul(a[..., ::2], b[..., ::2, :])


FORMS = {"nn": (_nn, lambda m, n, k: ((m, k), (k, n))), "tn": (_tn, lambda m, n, k: ((k, m), (k, n))),
         "nt": (_nt, lambda m, n, k: ((m, k), (n, k))),
         "strided": (_every_other, lambda m, n, k: ((m, 2 * k), (2 * k, n))),
         "reversed": (lambda a, b: np.matmul(np.flip(a, axis=a.ndim - 2), b), lambda m, n, k: ((m, k), (k, n)))}
SIZES = [(1, 1, 1, 1), (1, 1, 300, 700), (1, 64, 64, 32), (3, 65, 67, 33), (2, 17, 130, 257), (1, 200, 96, 1300),
         (5, 7, 16, 64), (1, 129, 1000, 31)]


@pytest.mark.gpu
@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("batch,M,N,K", SIZES)
@pytest.mark.parametrize("types", [("float32", "float32"), ("float16", "float32"), ("float32", "bfloat16")])
def test_products_match_float64(gpu, form, batch, M, N, K, types):
    print(f"dot {form} {batch}x{M}x{N}x{K} {types}", flush=True)
    fn, shapes = FORMS[form]
    rng = np.random.default_rng(M + N + K)
    arrays, exact = [], []
    for sh, d in zip(shapes(M, N, K), types):
        x = rng.standard_normal((batch,) + sh if batch > 1 else sh).astype(np.float32)
        y = dt.to_bf16(x) if d == "bfloat16" else x.astype(d)
        arrays.append(y)
        exact.append((dt.to_float32(y) if d == "bfloat16" else y).astype(np.float64))
    got = np.asarray(baremetal_jit(fn)(*arrays))
    assert got.dtype == np.float32
    ref, terms = fn(*exact), fn(*(np.abs(e) for e in exact))
    # fp32 sums of K exact or once-rounded products: at most K + 1 roundings
    # of 2^-24 of the terms' sizes, in practice their square root; the range
    # planes add no more
    bound = 2.0 ** -24 * (8 + 4 * np.sqrt(K)) * terms + 1e-30
    worst = float(np.max(np.abs(got - ref) / bound))
    assert worst <= 1.0


@pytest.mark.gpu
def test_small_and_special_values(gpu):
    """Subnormal operands and results, signed zeros, infinities and NaN."""
    a = np.array([[1e-40, 2e-39], [np.inf, 1.0], [np.nan, 0.0], [0.0, -0.0]], np.float32)
    b = np.array([[1.0, 2.0, 0.5], [3.0, 0.25, -1.0]], np.float32)
    got = np.asarray(baremetal_jit(_nn)(a, b))
    ref = (a.astype(np.float64) @ b).astype(np.float32)
    np.testing.assert_allclose(got[0], ref[0], rtol=0, atol=2e-45)
    np.testing.assert_array_equal(got[1:], ref[1:])


def test_ranges_and_load_modes():
    for batch, M, N, K in SIZES + [(1, 200, 1024, 3072), (1, 1, 8192, 2048), (1, 4096, 4096, 64), (1, 8, 8, 0)]:
        ks, kc = G.dot_split(batch, M, N, K)
        assert kc % 32 == 0 and ks >= 1 and (ks - 1) * kc < max(K, 1) <= ks * kc
    assert G.dot_split(1, 4096, 4096, 4096)[0] == 1 and G.dot_split(1, 200, 1024, 3072)[0] > 1
    # aligned and contiguous along k; along rows; a misaligned base, row or
    # batch stride; no unit stride
    assert G._dot_mode(256, 4, 64, 1, 4096, 10, 64, 2) == 1
    assert G._dot_mode(256, 4, 1, 64, 4096, 8, 10, 2) == 2
    assert G._dot_mode(260, 4, 64, 1, 4096, 10, 64, 2) == 0
    assert G._dot_mode(256, 4, 66, 1, 4096, 10, 64, 2) == 0
    assert G._dot_mode(256, 4, 64, 1, 4098, 10, 64, 2) == 0
    assert G._dot_mode(256, 4, 64, 1, 4096, 10, 63, 2) == 0
    assert G._dot_mode(256, 2, 64, 2, 0, 10, 64, 1) == 0
    assert G._dot_mode(256, 4, 65, 1, 0, 1, 64, 1) == 1
    assert G._dot_span(4, 64, 1, 10, 64) == 4 * 640 and G._dot_span(4, -64, 1, 10, 64) > 2**31


WIDE = [(1, 1, 128, 32), (2, 17, 130, 257), (1, 32, 384, 64), (3, 5, 900, 31), (1, 9, 65, 1100)]


@pytest.mark.gpu
@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("batch,M,N,K", WIDE)
def test_wide_tiles_match_float64(gpu, form, batch, M, N, K):
    """Sizes the 32 x 128 tiles take (fp32 pairs): every load mode, edges of
    both sides, ranges."""
    test_products_match_float64(gpu, form, batch, M, N, K, ("float32", "float32"))


def test_tile_choice():
    assert all(G.dot_tile(M, N, True) == (32, 128) for _, M, N, _ in WIDE)
    assert G.dot_tile(2, 1024, False) == (64, 64) and G.dot_tile(1, 64, True) == (64, 64)
    assert G.dot_tile(33, 4096, True) == (64, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("batch,M,N,K", sorted(set(SIZES + WIDE)))
@pytest.mark.parametrize("types", [("float32", "float32"), ("float16", "float32"), ("float32", "bfloat16")])
def test_matrix_core_form_at_small_sizes(gpu, monkeypatch, form, batch, M, N, K, types):
    """nk_dot_f32 at the sizes that dot_small leaves to nk_dot: the same edges
    of tiles, stages and load modes."""
    monkeypatch.setattr(G, "dot_small", lambda *a: False)
    monkeypatch.setitem(globals(), "baremetal_jit", _uncached)
    test_products_match_float64(gpu, form, batch, M, N, K, types)


def _uncached(fn):
    def call(*args):
        dk = DeviceKernel.compile_and_load(fn, *args, name="dot_small_off", use_cached_if_exists=False)
        symbols = [l.symbol for st in dk.plan.steps for l in st.launches(lambda v: 1 << 40)]
        assert "nk_dot" not in symbols or fn is FORMS["reversed"][0]
        ins = {n: DeviceTensor.from_numpy(a, name=n) for n, a in zip(dk.input_tensors_info, args)}
        return dk(ins)["output0"].numpy()
    return call


@pytest.mark.parametrize("batch,M,N,K,d,symbol", [
    (4096, 16, 16, 16, "float32", "nk_dot"), (1, 16, 16, 8192, "float32", "nk_dot_f32_f1_f2"),
    (4096, 17, 17, 4, "float32", "nk_dot"), (4096, 32, 64, 64, "float32", "nk_dot_f32_f1_f2"),
    (1, 64, 64, 64, "float16", "nk_dot"), (1, 64, 64, 64, "float32", "nk_dot_f32_f1_f2"),
    (1, 33, 33, 33, "float32", "nk_dot"), (512, 33, 33, 33, "float32", "nk_dot_f32_f0_f0"),
    (512, 33, 33, 17, "float16", "nk_dot_f32_h0_h0"), (1, 64, 64, 512, "float16", "nk_dot_f32_h1_h2"),
    (1, 8, 8, 0, "float32", "nk_dot")])
def test_small_products_keep_the_small_tiles(batch, M, N, K, d, symbol):
    plan = lower(NKIPyKernel.trace(_nn).specialize(np.zeros((batch, M, K), d), np.zeros((batch, K, N), d)))
    assert plan.steps[0].launches(lambda v: 1 << 40)[0].symbol == symbol
