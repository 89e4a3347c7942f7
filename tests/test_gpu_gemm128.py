"""The 128 x 128-tile GEMM kernels (gemm128.hip) on the GPU against the
256-tile kernels and, through them, the fp32 reference: sizes around the edges
of tiles, waves, MFMA tiles and K stages, every weight layout and epilogue,
and the K-range form with its reduction."""

import numpy as np
import pytest

from nkipy_amd.core import dtypes as dt
from nkipy_amd.dispatch import launchers as LA
from nkipy_amd.runtime import DeviceTensor
from oracle import numerics as N

pytestmark = pytest.mark.gpu

FORMS = [("nn", dt.bfloat16), ("nt", dt.bfloat16), ("nt", dt.float8_e4m3fn)]
SIZES = [(1, 8, 16), (33, 136, 80), (128, 128, 64), (129, 264, 208), (200, 64, 1056), (300, 520, 336)]


def _operands(rng, M, Nn, K, layout, bd):
    x = N.bf16_round(rng.standard_normal((M, K)))
    shape = (K, Nn) if layout == "nn" else (Nn, K)
    if bd == dt.bfloat16:
        w = N.bf16_round(rng.standard_normal(shape) / np.sqrt(K))
        return x, w, dt.to_bf16(w), None
    codes = rng.integers(0, 256, shape).astype(np.uint8)
    codes[(codes & 0x7f) == 0x7f] = 0  # no NaN codes
    scale = (rng.uniform(0.5, 1.5, Nn) / (100 * np.sqrt(K))).astype(np.float32)
    w = N.e4m3fn_decode(codes) * scale[:, None]
    return x, w, codes.view(dt.float8_e4m3fn), scale


def _dev(a):
    return DeviceTensor.from_numpy(a) if a is not None else None


def _clear(*tensors):
    """NaN everywhere, so that a launch under test has to write every element
    (and, in a workspace, every element that it reads)."""
    for t in tensors:
        t.write_from_numpy(np.full(t.nbytes, 0xff, np.uint8).view(t.dtype).reshape(t.shape))


def _check(got, ref, terms, rounded=0.0):
    # bf16 rounding of the result and of a value `rounded` on the way (each at
    # most 2^-8 of it) and fp32 sums whose terms' sizes add up to `terms`
    bound = 2.0 ** -7 * np.abs(ref) + 2.0 ** -7 * np.abs(rounded) + 2.0 ** -18 * terms
    worst = float(np.max(np.abs(got - ref) / bound))
    assert worst <= 1.0


@pytest.mark.parametrize("kh", [False, True])
@pytest.mark.parametrize("layout,bd", FORMS)
@pytest.mark.parametrize("M,Nn,K", SIZES)
def test_plain_bias_residual_and_ranges(gpu, M, Nn, K, layout, bd, kh):
    print(f"gemm128 kh={kh} {layout} {dt.name(bd)} {M}x{Nn}x{K}", flush=True)
    rng = np.random.default_rng(M * Nn + K)
    x, w, wd, scale = _operands(rng, M, Nn, K, layout, bd)
    bias, resid = N.bf16_round(rng.standard_normal(Nn)), N.bf16_round(rng.standard_normal((M, Nn)))
    tx, tw, ts, tb, tr = (_dev(a) for a in (dt.to_bf16(x), wd, scale, dt.to_bf16(bias), dt.to_bf16(resid)))
    prod = x.astype(np.float64) @ (w if layout == "nn" else w.T).astype(np.float64)
    terms = np.abs(x).astype(np.float64) @ np.abs(w if layout == "nn" else w.T).astype(np.float64)
    out = DeviceTensor.empty((M, Nn), dt.bfloat16)
    kw = dict(layout=layout, b_dtype=bd, c_dtype=dt.bfloat16, scale_ptr=ts.ptr if ts else 0, kh=kh)
    _clear(out)
    LA.gemm(tx.ptr, tw.ptr, out.ptr, M, Nn, K, tile=128, bias_ptr=tb.ptr, resid_ptr=tr.ptr, **kw).run(gpu)
    gpu.sync()
    _check(dt.to_float32(out.numpy()), prod + bias + resid, terms + 4)
    ks = 1 if K <= 64 else min(3, -(-K // 64))
    kc = -(-(-(-K // ks)) // 64) * 64
    ks = -(-K // kc)
    ws = DeviceTensor.empty((ks, M, Nn), np.float32)
    _clear(out, ws)
    for l in LA.gemm_splitk(tx.ptr, tw.ptr, out.ptr, M, Nn, K, split=(ks, kc), ws_ptr=ws.ptr,
                            resid_ptr=tr.ptr, round_before_resid=True, **kw):
        l.run(gpu)
    gpu.sync()
    _check(dt.to_float32(out.numpy()), N.bf16_round(prod) + resid, terms + 4, rounded=prod)


@pytest.mark.parametrize("kh", [False, True])
@pytest.mark.parametrize("layout,bd", FORMS)
@pytest.mark.parametrize("M,Nn,K", SIZES)
def test_swiglu(gpu, M, Nn, K, layout, bd, kh):
    print(f"gemm128 swiglu kh={kh} {layout} {dt.name(bd)} {M}x{Nn}x{K}", flush=True)
    rng = np.random.default_rng(M + Nn * K)
    x, w, wd, scale = _operands(rng, M, Nn, K, layout, bd)
    _, u, ud, uscale = _operands(rng, M, Nn, K, layout, bd)
    tx, tw, ts, tu, tus = (_dev(a) for a in (dt.to_bf16(x), wd, scale, ud, uscale))
    g, v = (x.astype(np.float64) @ (m if layout == "nn" else m.T).astype(np.float64) for m in (w, u))
    ref = g / (1 + np.exp(-g)) * v
    out = DeviceTensor.empty((M, Nn), dt.bfloat16)
    kw = dict(layout=layout, b_dtype=bd, c_dtype=dt.bfloat16, scale_ptr=ts.ptr if ts else 0, up_ptr=tu.ptr,
              up_scale_ptr=tus.ptr if tus else 0, kh=kh)
    _clear(out)
    LA.gemm(tx.ptr, tw.ptr, out.ptr, M, Nn, K, tile=128, **kw).run(gpu)
    gpu.sync()
    _check(dt.to_float32(out.numpy()), ref, 8 * (1 + np.abs(g)) * (1 + np.abs(v)))
    kc = -(-(-(-K // 2)) // 64) * 64
    ks = -(-K // kc)
    ws = DeviceTensor.empty((2, ks, M, Nn), np.float32)
    _clear(out, ws)
    for l in LA.gemm_splitk(tx.ptr, tw.ptr, out.ptr, M, Nn, K, split=(ks, kc), ws_ptr=ws.ptr, **kw):
        l.run(gpu)
    gpu.sync()
    _check(dt.to_float32(out.numpy()), ref, 8 * (1 + np.abs(g)) * (1 + np.abs(v)))


@pytest.mark.parametrize("layout,bd", FORMS)
def test_rotary_equals_the_256_tile_kernel(gpu, layout, bd):
    """q / k heads rotated in the epilogue, value columns to C: the same
    products in the same K order give the 256-tile kernel's bits; the eight-
    wave form, which adds two interleaved sums, is within a rounding step of
    them."""
    B, S, K, nq, nk, nv = 3, 67, 208, 256, 128, 128
    M, Nn = B * S, nq + nk + nv
    print(f"gemm128 rope {layout} {dt.name(bd)}", flush=True)
    rng = np.random.default_rng(5)
    x, w, wd, scale = _operands(rng, M, Nn, K, layout, bd)
    ang = rng.uniform(0, 6, (S, 64))
    tx, tw, ts, tc, tsn = (_dev(a) for a in (dt.to_bf16(x), wd, scale, np.cos(ang).astype(np.float32),
                                             np.sin(ang).astype(np.float32)))
    got = []
    for opt in ({}, {"tile": 128, "kh": False}, {"tile": 128, "kh": True}, {"tile": 64}):
        q, k, c = (DeviceTensor.from_numpy(dt.to_bf16(np.zeros((M, n), np.float32))) for n in (nq, nk, Nn))
        rope = LA.GemmRope(tc.ptr, tsn.ptr, q.ptr, k.ptr, 64, S, nq, nk)
        LA.gemm(tx.ptr, tw.ptr, c.ptr, M, Nn, K, layout=layout, b_dtype=bd, c_dtype=dt.bfloat16,
                scale_ptr=ts.ptr if ts else 0, rope=rope, **opt).run(gpu)
        gpu.sync()
        got.append([dt.to_float32(t.numpy()) for t in (q, k, c)])
    for a, b, h, h64 in zip(*got):
        assert np.array_equal(a, b) and np.array_equal(h, h64)
        # a product moved by one rounding step (2^-8 of it) moves both halves' rotations
        worst = float(np.max(np.abs(h - a)) / np.max(np.abs(a)))
        assert worst <= 2.0 ** -7


@pytest.mark.parametrize("c_dtype", [dt.bfloat16, dt.float32])
@pytest.mark.parametrize("ks", [1, 2, 5, 9])
def test_reduction_forms_agree(gpu, ks, c_dtype):
    """Four outputs per thread and one wave per four ranges add the planes in
    the same order: the same bits, plain, biased and with a residual."""
    M, Nn = 37, 264
    rng = np.random.default_rng(ks)
    pl = rng.standard_normal((2, ks, M, Nn), dtype=np.float32)
    sc, bi = rng.uniform(0.5, 2, Nn).astype(np.float32), N.bf16_round(rng.standard_normal(Nn))
    planes, scale, bias = (DeviceTensor.from_numpy(a) for a in (pl, sc, dt.to_bf16(bi)))
    r = rng.standard_normal((M, Nn)).astype(np.float32)
    r = N.bf16_round(r) if c_dtype == dt.bfloat16 else r
    resid = DeviceTensor.from_numpy(dt.to_bf16(r) if c_dtype == dt.bfloat16 else r)
    out = DeviceTensor.empty((M, Nn), c_dtype)
    flags = LA.GEMM_BIAS | LA.GEMM_SCALE | LA.GEMM_RESID | LA.GEMM_RND_BIAS | LA.GEMM_RND_RESID
    for swiglu, fl in ((False, 0), (False, flags), (True, LA.GEMM_SCALE)):
        if swiglu and c_dtype != dt.bfloat16:
            continue
        args = LA.GemvArgs(0, 0, 0, out.ptr, bias.ptr, scale.ptr, scale.ptr, resid.ptr, planes.ptr, M, Nn, 64, 64,
                           Nn, Nn, ks, 64, fl, 0)
        got = []
        for least in (1 << 62, 0):
            saved, LA.REDUCE4_MIN = LA.REDUCE4_MIN, least
            try:
                l = LA._reduce_planes(args, c_dtype, swiglu)
            finally:
                LA.REDUCE4_MIN = saved
            assert bool(l.args.flags & LA.GEMV_OUT4) is (least == 0)
            _clear(out)
            l.run(gpu)
            gpu.sync()
            got.append(out.numpy().tobytes())
        assert got[0] == got[1]
        # fp32 sums of ks terms; the rounding of the result and, with the
        # epilogue, of the product and the biased product to bf16
        g, u = pl.astype(np.float64).sum(1)
        sums = 2.0 ** -22 * np.abs(pl).astype(np.float64).sum(1).max(0)
        last = 2.0 ** -8 if c_dtype == dt.bfloat16 else 2.0 ** -23
        if swiglu:
            ref = g * sc / (1 + np.exp(-g * sc)) * (u * sc)
            bound = last * np.abs(ref) + 8 * sums * (1 + np.abs(g)) * (1 + np.abs(u)) * sc * sc
        elif fl:
            p, b = g * sc, g * sc + bi
            ref = b + r
            bound = last * np.abs(ref) + 2.0 ** -8 * (np.abs(p) + np.abs(b)) + 4 * sums * sc
        else:
            ref, bound = g, last * np.abs(g) + sums
        o = out.numpy()
        o = dt.to_float32(o) if c_dtype == dt.bfloat16 else o
        assert np.all(np.abs(o - ref) <= bound + 1e-30)


@pytest.mark.parametrize("layout,bd", FORMS)
@pytest.mark.parametrize("M,Nn,K", [(1, 8, 16), (17, 136, 80), (32, 264, 1056), (33, 128, 592), (49, 200, 640),
                                    (64, 520, 1200)])
def test_few_row_tiles(gpu, M, Nn, K, layout, bd):
    """The 64- and 32-row forms: edges of the MFMA row tiles, rings shorter and
    longer than K, plain, over ranges and as a SwiGLU pair."""
    print(f"gemm128 few rows {layout} {dt.name(bd)} {M}x{Nn}x{K}", flush=True)
    rng = np.random.default_rng(M + Nn + K)
    x, w, wd, scale = _operands(rng, M, Nn, K, layout, bd)
    _, u, ud, uscale = _operands(rng, M, Nn, K, layout, bd)
    tx, tw, ts, tu, tus = (_dev(a) for a in (dt.to_bf16(x), wd, scale, ud, uscale))
    g, v = (x.astype(np.float64) @ (m if layout == "nn" else m.T).astype(np.float64) for m in (w, u))
    terms = np.abs(x).astype(np.float64) @ np.abs(w if layout == "nn" else w.T).astype(np.float64)
    out = DeviceTensor.empty((M, Nn), dt.bfloat16)
    kc = max(64, -(-(-(-K // 3)) // 64) * 64)
    ks = -(-K // kc)
    ws = DeviceTensor.empty((2, ks, M, Nn), np.float32)
    for kh in (64, 32) if M <= 32 else (64,):
        kw = dict(layout=layout, b_dtype=bd, c_dtype=dt.bfloat16, scale_ptr=ts.ptr if ts else 0, kh=kh)
        pair = dict(up_ptr=tu.ptr, up_scale_ptr=tus.ptr if tus else 0, **kw)
        for opt, ref, size in ((kw, g, terms), (pair, g / (1 + np.exp(-g)) * v, 8 * (1 + np.abs(g)) * (1 + np.abs(v)))):
            l = LA.gemm(tx.ptr, tw.ptr, out.ptr, M, Nn, K, tile=128, **opt)
            assert l.symbol.endswith(f"_kh{kh}")
            _clear(out)
            l.run(gpu)
            gpu.sync()
            _check(dt.to_float32(out.numpy()), ref, size)
            _clear(out, ws)
            for l in LA.gemm_splitk(tx.ptr, tw.ptr, out.ptr, M, Nn, K, split=(ks, kc), ws_ptr=ws.ptr, **opt):
                l.run(gpu)
            gpu.sync()
            _check(dt.to_float32(out.numpy()), ref, size)


@pytest.mark.parametrize("layout,bd", FORMS)
@pytest.mark.parametrize("M,Nn,K", [(65, 136, 80), (128, 264, 1056), (200, 128, 592), (321, 72, 640)])
def test_64_row_tiles(gpu, layout, bd, M, Nn, K):
    """Several 64-row tiles: plain with bias and residual, and as a SwiGLU
    pair."""
    print(f"gemm128 64-row tiles {layout} {dt.name(bd)} {M}x{Nn}x{K}", flush=True)
    rng = np.random.default_rng(M + Nn + K)
    x, w, wd, scale = _operands(rng, M, Nn, K, layout, bd)
    _, u, ud, uscale = _operands(rng, M, Nn, K, layout, bd)
    bias, resid = N.bf16_round(rng.standard_normal(Nn)), N.bf16_round(rng.standard_normal((M, Nn)))
    tx, tw, ts, tu, tus, tb, tr = (_dev(a) for a in (dt.to_bf16(x), wd, scale, ud, uscale, dt.to_bf16(bias),
                                                     dt.to_bf16(resid)))
    g, v = (x.astype(np.float64) @ (m if layout == "nn" else m.T).astype(np.float64) for m in (w, u))
    terms = np.abs(x).astype(np.float64) @ np.abs(w if layout == "nn" else w.T).astype(np.float64)
    out = DeviceTensor.empty((M, Nn), dt.bfloat16)
    kw = dict(layout=layout, b_dtype=bd, c_dtype=dt.bfloat16, scale_ptr=ts.ptr if ts else 0, tile=64)
    l = LA.gemm(tx.ptr, tw.ptr, out.ptr, M, Nn, K, bias_ptr=tb.ptr, resid_ptr=tr.ptr, **kw)
    assert l.symbol.endswith("_kh64") and l.grid[0] == -(-M // 64) * -(-Nn // 128)
    _clear(out)
    l.run(gpu)
    gpu.sync()
    _check(dt.to_float32(out.numpy()), g + bias + resid, terms + 4)
    _clear(out)
    LA.gemm(tx.ptr, tw.ptr, out.ptr, M, Nn, K, up_ptr=tu.ptr, up_scale_ptr=tus.ptr if tus else 0, **kw).run(gpu)
    gpu.sync()
    _check(dt.to_float32(out.numpy()), g / (1 + np.exp(-g)) * v, 8 * (1 + np.abs(g)) * (1 + np.abs(v)))
