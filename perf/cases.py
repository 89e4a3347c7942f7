"""Performance cases of the framework: the kernels a user's program calls,
through ``DeviceKernel``, over the sizes, types and directions in use.

Every case traces one of the package's NumPy kernels (or the language-model
head below, written the way such kernels are written), loads it once with its
tensors in device memory, as a program does, and then calls it.  Sizes follow
the package's own workloads (hidden 4096 with 32 / 8 heads of 128 and FFN
14336, smaller siblings of it, expert-sized MLPs, a 151936-token head) and
run down to single rows and through odd row counts, prompt lengths, cache
lengths and positions.  Layers of a stack and decode steps queue
(``sync=False``); calls whose result the host needs wait, as they do by
default.

Case kinds and the parameters ``draw`` varies:

  softmax          rows, n, dtype
  residual_norm    rows, hidden, dtype
  swiglu_mlp       rows, hidden, ffn (bf16, two weights)
  feedforward      rows, hidden, ffn, dtype (bf16 or fp32, one gate_up weight)
  linear_attention batch, heads, seq (bf16, head dim 128)
  fp8_attention    batch, seq, hidden, heads, kv_heads (prefill block)
  fp8_mlp          rows, hidden, ffn
  fp8_layer        batch, seq, hidden, heads, kv_heads, ffn (whole layer)
  qwen3_prefill    batch, seq, cache, hidden, heads, kv_heads (whole attention layer)
  qwen3_decode     batch, cache, pos, hidden, heads, kv_heads (the same, one token)
  lm_head          batch, hidden, vocab (logits and the greedy token)
"""

import math

import numpy as np
import torch

from nkipy_amd import kernels as K
from nkipy_amd.core import tensor_apis
from nkipy_amd.kernels import qwen3
from nkipy_amd.runtime import DeviceKernel, DeviceTensor

HEAD_DIM = 128
ROPE_THETA = 5.0e5       # the fp8 layer
QWEN_ROPE_BASE = 1000000
EPS = 1e-6
LAYER_EPS = 1e-5         # the fp8 layer's default

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}


def lm_head_kernel(h, norm_weight, lm_head_weight, norm_eps):
    """Logits of the last position and the greedy token: qwen3.greedy_sampling
    for a program that also keeps the logits (log-probabilities, sampling)."""
    h = K.rmsnorm_kernel(h, norm_weight, norm_eps)
    logits = h[:, -1, :] @ lm_head_weight
    _, next_id = tensor_apis.topk(logits, k=1, axis=1)
    return logits, next_id


# ---------------------------------------------------------------------------
# The listed cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The first kernel of the README on a small batch of scores: a call
        # whose launch and wait are most of its time.
        {"name": "softmax_small", "kind": "softmax", "rows": 32, "n": 1000, "dtype": "f32"},
        # Residual add and norm between two layers, a large prefill.
        {"name": "residual_norm", "kind": "residual_norm", "rows": 8192, "hidden": 4096, "dtype": "bf16"},
        # The MLP of a bf16 model, a full prefill chunk.
        {"name": "swiglu_mlp", "kind": "swiglu_mlp", "rows": 4096, "hidden": 4096, "ffn": 14336},
        # A Qwen3-style fused gate_up MLP, a short prompt of 300 tokens.
        {"name": "feedforward_bf16", "kind": "feedforward", "rows": 300, "hidden": 4096, "ffn": 12288,
         "dtype": "bf16"},
        # The same kernel on fp32 arrays, NumPy's everyday type (an embedding
        # model's MLP on 200 tokens).
        {"name": "feedforward_f32", "kind": "feedforward", "rows": 200, "hidden": 1024, "ffn": 3072,
         "dtype": "f32"},
        # Linear attention over long sequences.
        {"name": "linear_attention", "kind": "linear_attention", "batch": 4, "heads": 16, "seq": 8192},
        # Attention block of the fp8 model, two prompts of a length nobody
        # rounded.
        {"name": "fp8_attention_ragged", "kind": "fp8_attention", "batch": 2, "seq": 1000, "hidden": 4096,
         "heads": 32, "kv_heads": 8},
        # MLP block of the fp8 model for a batch of decode tokens.
        {"name": "fp8_mlp_decode", "kind": "fp8_mlp", "rows": 24, "hidden": 4096, "ffn": 14336},
        # The whole fp8 decoder layer, eight prompts of 2048 tokens (the
        # largest case).
        {"name": "fp8_layer", "kind": "fp8_layer", "batch": 8, "seq": 2048, "hidden": 4096, "heads": 32,
         "kv_heads": 8, "ffn": 14336},
        # Qwen3 attention layer, prefill of one prompt into a KV cache.
        {"name": "qwen3_prefill", "kind": "qwen3_prefill", "batch": 1, "seq": 1500, "cache": 2048, "hidden": 4096,
         "heads": 32, "kv_heads": 8},
        # The same layer generating: one token for each of eight sequences.
        {"name": "qwen3_decode", "kind": "qwen3_decode", "batch": 8, "cache": 4096, "pos": 4000, "hidden": 4096,
         "heads": 32, "kv_heads": 8},
        # The end of every decode step: final norm, logits, greedy token.
        {"name": "lm_head", "kind": "lm_head", "batch": 8, "hidden": 4096, "vocab": 151936},
    ]


def _log(rng, lo, hi):
    """An integer from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.499)))))))


_HEADS = [(4096, 32, 8), (2048, 16, 8), (2048, 16, 2), (1024, 8, 8), (5120, 40, 8)]
_FFN = [(4096, 14336), (4096, 12288), (2048, 6144), (2048, 1536), (1024, 3072)]
MOST_FLOPS = 2e12  # of a drawn case (the largest listed one has 7.4e12)


def draw(rng):
    while True:
        c = _draw(rng)
        if _flops(c) <= MOST_FLOPS:
            return c


def _draw(rng):
    kind = rng.choice(["softmax", "residual_norm", "swiglu_mlp", "feedforward", "feedforward", "linear_attention",
                       "fp8_attention", "fp8_mlp", "fp8_layer", "qwen3_prefill", "qwen3_decode", "lm_head"])
    c = {"kind": kind}
    if kind == "softmax":
        n = _log(rng, 16, 32768)
        if rng.random() < 0.5:  # half of the rows in whole 16-byte pieces
            n = max(16, n // 8 * 8)
        c.update(rows=_log(rng, 1, min(8192, 2 ** 25 // n)), n=n, dtype=rng.choice(["f32", "f32", "bf16", "f16"]))
    elif kind == "residual_norm":
        c.update(rows=_log(rng, 1, 16384), hidden=64 * _log(rng, 8, 128), dtype=rng.choice(["bf16", "bf16", "f32", "f16"]))
    elif kind == "swiglu_mlp":
        hidden, ffn = rng.choice(_FFN)
        c.update(rows=_log(rng, 1, 4096), hidden=hidden, ffn=ffn)
    elif kind == "feedforward":
        dtype = rng.choice(["bf16", "f32"])
        hidden, ffn = rng.choice(_FFN if dtype == "bf16" else _FFN[2:])
        c.update(rows=_log(rng, 1, 4096 if dtype == "bf16" else 1024), hidden=hidden, ffn=ffn, dtype=dtype)
    elif kind == "linear_attention":
        c.update(batch=rng.choice([1, 2, 3, 4]), heads=rng.choice([4, 6, 8, 12, 16]), seq=64 * _log(rng, 2, 160))
    elif kind in ("fp8_attention", "fp8_layer"):
        hidden, heads, kv = rng.choice(_HEADS)
        seq = _log(rng, 8, 2048)
        c.update(batch=_log(rng, 1, max(1, min(8, 4096 // seq))), seq=seq, hidden=hidden, heads=heads, kv_heads=kv)
        if kind == "fp8_layer":
            c["ffn"] = 3 * hidden
    elif kind == "fp8_mlp":
        hidden, ffn = rng.choice(_FFN)
        c.update(rows=_log(rng, 1, 4096), hidden=hidden, ffn=ffn)
    elif kind == "qwen3_prefill":
        hidden, heads, kv = rng.choice(_HEADS)
        seq = _log(rng, 8, 2048)
        c.update(batch=1 if seq > 512 else rng.choice([1, 2, 4]), seq=seq,
                 cache=256 * -(-rng.randint(seq, max(seq, 2048)) // 256), hidden=hidden, heads=heads, kv_heads=kv)
    elif kind == "qwen3_decode":
        hidden, heads, kv = rng.choice(_HEADS)
        cache = 256 * _log(rng, 2, 16)
        c.update(batch=_log(rng, 1, 64), cache=cache, pos=rng.randint(cache // 4, cache - 1), hidden=hidden,
                 heads=heads, kv_heads=kv)
    else:
        c.update(batch=_log(rng, 1, 32), hidden=rng.choice([1024, 2048, 4096]), vocab=rng.choice([32000, 128256, 151936]))
    return c


# ---------------------------------------------------------------------------
# What a program has in hand before the call
# ---------------------------------------------------------------------------
class _Memory:
    """A DeviceTensor's buffer as torch sees it (no copy); a torch view keeps
    this object, and with it the buffer, alive."""

    _TYPES = {1: "|u1", 2: "<i2", 4: "<f4"}

    def __init__(self, t, itemsize):
        self.owner = t
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": self._TYPES[itemsize], "data": (t.ptr, False),
                                         "version": 2}


def _as_torch(t, dtype):
    return torch.as_tensor(_Memory(t, dtype.itemsize), device="cuda").view(dtype)


class _Inputs:
    """Seeded inputs on the GPU, in their order of creation."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def normal(self, shape, std=1.0, dtype=torch.bfloat16):
        return (torch.randn(shape, generator=self.gen, device="cuda") * std).to(dtype)

    def uniform(self, shape, lo, hi, dtype=torch.bfloat16):
        return (torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo).to(dtype)

    def integers(self, shape, n):
        return torch.randint(0, n, shape, generator=self.gen, device="cuda")

    def fp8(self, out, inp, std=0.02):
        """An (out, in) weight quantized to e4m3 with per-output-channel scales."""
        w = torch.randn((out, inp), generator=self.gen, device="cuda") * std
        s = w.abs().amax(1) / 448.0
        return (w / s[:, None]).to(torch.float8_e4m3fn), s


def _kernel_of(c):
    """(kernel, arguments after the tensors, keyword arguments)."""
    kind = c["kind"]
    if kind == "softmax":
        return K.softmax_kernel, (), {}
    if kind == "residual_norm":
        return K.residual_rmsnorm_kernel, (EPS,), {}
    if kind == "swiglu_mlp":
        return K.swiglu_mlp_kernel, (), {}
    if kind == "feedforward":
        return K.feedforward_kernel, (), {}
    if kind == "linear_attention":
        return K.chunked_linear_attention_kernel, (), {}
    if kind == "fp8_attention":
        return K.attention_block_fp8, (), {"n_heads": c["heads"], "n_kv_heads": c["kv_heads"]}
    if kind == "fp8_mlp":
        return K.mlp_block_fp8, (), {}
    if kind == "fp8_layer":
        return K.llama_decoder_layer_fp8, (), {"n_heads": c["heads"], "n_kv_heads": c["kv_heads"]}
    if kind == "lm_head":
        return lm_head_kernel, (EPS,), {}
    return None  # qwen3: the arguments are interleaved


def _tensors(c, seed):
    """Named input tensors of the case, in the kernel's argument order."""
    r, kind = _Inputs(seed), c["kind"]
    if kind == "softmax":
        return {"x": r.normal((c["rows"], c["n"]), 4.0, TORCH[c["dtype"]])}
    if kind == "residual_norm":
        t, sh = TORCH[c["dtype"]], (c["rows"], c["hidden"])
        return {"x": r.normal(sh, 1.0, t), "residual": r.normal(sh, 1.0, t), "weight": r.uniform(sh[1:], 0.5, 1.5, t)}
    if kind == "swiglu_mlp":
        h, f = c["hidden"], c["ffn"]
        return {"x": r.normal((c["rows"], h)), "w_gate": r.normal((h, f), 0.02), "w_up": r.normal((h, f), 0.02),
                "w_down": r.normal((f, h), 0.02)}
    if kind == "feedforward":
        h, f, t = c["hidden"], c["ffn"], TORCH[c["dtype"]]
        return {"x": r.normal((c["rows"], h), 1.0, t), "gate_up_weight": r.normal((h, 2 * f), 0.02, t),
                "down_weight": r.normal((f, h), 0.02, t)}
    if kind == "linear_attention":
        sh = (c["batch"], c["heads"], c["seq"], HEAD_DIM)
        return {n: r.normal(sh, HEAD_DIM ** -0.5) for n in ("q", "k", "v")}
    if kind == "lm_head":
        h, v = c["hidden"], c["vocab"]
        w = r.normal((h, v), 0.02)
        # a trained head's logits have a leader: each hidden state points at
        # one token's column
        lead = r.integers((c["batch"],), v)
        x = r.normal((c["batch"], 1, h)) + (w[:, lead].T.float()[:, None, :] * 20.0).to(torch.bfloat16)
        return {"h": x, "norm_weight": r.uniform((h,), 0.5, 1.5), "lm_head_weight": w}
    h = c["hidden"]
    if kind in ("fp8_attention", "fp8_mlp", "fp8_layer"):
        d = {}
        if kind == "fp8_mlp":
            d["z"] = r.normal((c["rows"], h))
        else:
            nq, hq = (c["heads"] + 2 * c["kv_heads"]) * HEAD_DIM, c["heads"] * HEAD_DIM
            d["x"] = r.normal((c["batch"], c["seq"], h))
            d["norm_weight" if kind == "fp8_attention" else "attn_norm_weight"] = r.uniform((h,), 0.5, 1.5)
            d["wqkv"], d["wqkv_scale"] = r.fp8(nq, h)
            d["wo"], d["wo_scale"] = r.fp8(h, hq)
        if kind != "fp8_attention":
            f = c["ffn"]
            d["norm_weight" if kind == "fp8_mlp" else "mlp_norm_weight"] = r.uniform((h,), 0.5, 1.5)
            for n, o, i in (("w_gate", f, h), ("w_up", f, h), ("w_down", h, f)):
                d[n], d[n + "_scale"] = r.fp8(o, i)
        return d
    # qwen3: heads, a cache with its earlier tokens (or stale rows, for a
    # prefill) and the token's position
    nq, hq = (c["heads"] + 2 * c["kv_heads"]) * HEAD_DIM, c["heads"] * HEAD_DIM
    cache = (c["batch"], c["cache"], c["kv_heads"], HEAD_DIM)
    d = {"x": r.normal((c["batch"], c.get("seq", 1), h)), "qkv_weight": r.normal((h, nq), 0.02),
         "q_norm_weight": r.uniform((HEAD_DIM,), 0.5, 1.5), "k_norm_weight": r.uniform((HEAD_DIM,), 0.5, 1.5),
         "cache_k": r.normal(cache), "cache_v": r.normal(cache)}
    if kind == "qwen3_decode":
        d["start_pos"] = torch.full((1,), c["pos"], dtype=torch.int32, device="cuda")
    d["o_weight"] = r.normal((hq, h), 0.02)
    return d


_NUMPY = {torch.float32: "float32", torch.float16: "float16", torch.int32: "int32", torch.bfloat16: "bfloat16",
          torch.float8_e4m3fn: "float8_e4m3fn"}


def prepare(case, seed):
    c = case
    host = _tensors(c, seed)
    dev = {}
    for n, t in host.items():
        dev[n] = DeviceTensor.empty(tuple(t.shape), _NUMPY[t.dtype], name=n)
        _as_torch(dev[n], t.dtype).copy_(t)
    del host
    found = _kernel_of(c)
    if found is not None:
        kernel, rest, kw = found
        args = tuple(dev.values()) + rest
    else:
        kernel, kw = qwen3.qwen3_attention_kernel, {}
        args = (dev["x"], dev["qkv_weight"], dev["q_norm_weight"], dev["k_norm_weight"], EPS, c["heads"], HEAD_DIM,
                c["kv_heads"], dev["cache_k"], dev["cache_v"], dev.get("start_pos"), dev["o_weight"])
    dk = DeviceKernel.compile_and_load(kernel, *args, **kw)
    alias = ".must_alias_input"
    inputs = {n: dev[n.split(alias)[0]] for n in dk.input_tensors_info}
    outputs, views = {}, {}
    for n, info in dk.output_tensors_info.items():
        outputs[n] = dev[n] if n in dev else DeviceTensor.empty(tuple(info.shape), info.dtype, name=n)
        views[n] = _as_torch(outputs[n], {"uint32": torch.int32}.get(info.dtype) or getattr(torch, info.dtype))
    # results the host waits for; layers of a stack and decode steps queue
    sync = c["kind"] in ("softmax", "linear_attention", "lm_head") or c.get("dtype") == "f32"
    torch.cuda.synchronize()
    return {"kernel": dk, "inputs": inputs, "outputs": outputs, "views": views, "sync": sync}


def run(state):
    state["kernel"](state["inputs"], state["outputs"], sync=state["sync"])
    return state["views"]


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------
def _flops(c):
    kind = c["kind"]
    if kind in ("softmax", "residual_norm"):
        return 5 * c["rows"] * c.get("n", c.get("hidden"))
    if kind in ("swiglu_mlp", "feedforward", "fp8_mlp"):
        return 6 * c["rows"] * c["hidden"] * c["ffn"]
    if kind == "linear_attention":
        # per chunk of 64: scores, weighted values, state update, state read
        n = c["batch"] * c["heads"] * c["seq"]
        return n * 4 * HEAD_DIM * (64 + HEAD_DIM)
    if kind == "lm_head":
        return 2 * c["batch"] * c["hidden"] * c["vocab"]
    h, hq, hkv = c["hidden"], c["heads"] * HEAD_DIM, c["kv_heads"] * HEAD_DIM
    if kind == "qwen3_decode":
        return c["batch"] * (2 * h * (hq + 2 * hkv) + 2 * hq * h + 4 * hq * (c["pos"] + 1))
    m = c["batch"] * c["seq"]
    # causal: query i sees i + 1 keys
    f = 2 * m * h * (hq + 2 * hkv) + 2 * m * hq * h + 2 * c["batch"] * hq * c["seq"] * (c["seq"] + 1)
    if kind == "fp8_layer":
        f += 6 * m * h * c["ffn"]
    return f


def work(case):
    c, kind = case, case["kind"]
    if kind == "softmax":
        b = 2 * c["rows"] * c["n"] * SIZE[c["dtype"]]
    elif kind == "residual_norm":
        b = (3 * c["rows"] + 1) * c["hidden"] * SIZE[c["dtype"]]
    elif kind in ("swiglu_mlp", "feedforward"):
        b = (2 * c["rows"] * c["hidden"] + 3 * c["hidden"] * c["ffn"]) * SIZE[c.get("dtype", "bf16")]
    elif kind == "linear_attention":
        b = 4 * c["batch"] * c["heads"] * c["seq"] * HEAD_DIM * 2
    elif kind == "lm_head":
        b = 2 * (c["batch"] * c["hidden"] + c["hidden"] * c["vocab"] + c["batch"] * c["vocab"])
    elif kind == "fp8_mlp":
        b = 4 * c["rows"] * c["hidden"] + 3 * c["hidden"] * c["ffn"]
    else:
        h, hq, hkv = c["hidden"], c["heads"] * HEAD_DIM, c["kv_heads"] * HEAD_DIM
        weights = h * (hq + 2 * hkv) + hq * h
        m = c["batch"] * c.get("seq", 1)
        if kind == "qwen3_decode":
            # the weights, the cached keys and values up to pos, the new rows
            b = 2 * weights + 4 * m * h + 4 * c["batch"] * (c["pos"] + 2) * hkv
        elif kind == "qwen3_prefill":
            b = 2 * weights + 4 * m * h + 4 * m * hkv
        else:
            b = weights + 4 * m * h + (3 * h * c["ffn"] if kind == "fp8_layer" else 0)
    return {"bytes": b, "flops": _flops(c)}


def tolerance(case):
    """Relative error of another correct implementation: the order of 32-bit
    sums, and for 16-bit results the last place of what is stored on the way
    (a rounding that falls the other way); about four times the difference
    seen against the 64-bit evaluation, of which the result's own rounding is
    the larger part."""
    kind, dtype = case["kind"], case.get("dtype", "bf16")
    if dtype == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if kind in ("softmax", "residual_norm"):
        return {"rel": 1e-2 if dtype == "bf16" else 1.5e-3, "max": 0.1}
    if kind == "lm_head":
        return {"rel": 1e-2, "max": 0.2, "differ": 0.0}
    return {"rel": 1.2e-2, "max": 0.5}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _norm64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _silu64(x):
    return x / (1 + torch.exp(-x))


def _rope64(x, base):
    """Split-half rotation of (B, S, H, D), positions 0..S-1 of dim 1."""
    half = x.shape[-1] // 2
    return _rope64_at(x, torch.arange(x.shape[1], device=x.device, dtype=torch.float64), base, half)


def _rope64_at(x, pos, base, half):
    inv = base ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    ang = pos[:, None] * inv[None]
    c, s = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]
    x0, x1 = x[..., :half], x[..., half:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)


def _causal64(q, k, v):
    """q (B, S, Hq, D), k / v (B, S, Hkv, D) -> (B, S, Hq * D), one sequence
    and KV head at a time."""
    B, S, hq, d = q.shape
    rep = hq // k.shape[2]
    out = torch.empty_like(q)
    hidden = torch.triu(torch.ones((S, S), dtype=torch.bool, device=q.device), 1)
    for b in range(B):
        for g in range(k.shape[2]):
            for h in range(g * rep, (g + 1) * rep):
                s = (q[b, :, h] @ k[b, :, g].T.contiguous()) / math.sqrt(d)
                out[b, :, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[b, :, g].contiguous()
    return out.reshape(B, S, hq * d)


def _split_heads(x, heads, kv):
    B, S, _ = x.shape
    q, k, v = torch.split(x, [heads * HEAD_DIM, kv * HEAD_DIM, kv * HEAD_DIM], -1)
    return (q.reshape(B, S, heads, HEAD_DIM), k.reshape(B, S, kv, HEAD_DIM), v.reshape(B, S, kv, HEAD_DIM))


def exact(case, seed):
    c, kind = case, case["kind"]
    t = {n: v if v.dtype == torch.int32 else v.to(torch.float32).double() for n, v in _tensors(c, seed).items()}
    mat = lambda x, n: x @ (t[n] * t[n + "_scale"][:, None]).T.contiguous()  # an fp8 weight
    if kind == "softmax":
        return {"output0": torch.softmax(t["x"], -1)}
    if kind == "residual_norm":
        return {"output0": _norm64(t["x"] + t["residual"], t["weight"], EPS)}
    if kind == "swiglu_mlp":
        return {"output0": (_silu64(t["x"] @ t["w_gate"]) * (t["x"] @ t["w_up"])) @ t["w_down"]}
    if kind == "feedforward":
        g, u = (t["x"] @ t["gate_up_weight"]).chunk(2, -1)
        return {"output0": (_silu64(g) * u) @ t["down_weight"]}
    if kind == "linear_attention":
        phi = lambda x: torch.where(x > 0, x + 1, torch.exp(x))
        q, k, v = phi(t["q"]), phi(t["k"]), t["v"]
        out = torch.empty_like(v)
        mask = torch.tril(torch.ones((64, 64), dtype=torch.float64, device=v.device))
        B, H, T, D = q.shape
        state = torch.zeros((B * H, D, D), dtype=torch.float64, device=v.device)
        z = torch.zeros((B * H, D, 1), dtype=torch.float64, device=v.device)
        for i in range(0, T, 64):
            a, b, w = (x[:, :, i:i + 64].reshape(B * H, 64, D) for x in (q, k, v))
            bt = b.transpose(1, 2).contiguous()
            sc = torch.bmm(a, bt) * mask
            num, den = torch.bmm(a, state) + torch.bmm(sc, w), torch.bmm(a, z) + sc.sum(-1, keepdim=True)
            out[:, :, i:i + 64] = (num / den).reshape(B, H, 64, D)
            state, z = state + torch.bmm(bt, w), z + bt.sum(-1, keepdim=True)
        return {"output0": out}
    if kind == "lm_head":
        logits = _norm64(t["h"], t["norm_weight"], EPS)[:, -1] @ t["lm_head_weight"]
        return {"output0": logits, "output1": None}
    if kind in ("fp8_attention", "fp8_mlp", "fp8_layer"):
        z = t.get("z")
        if kind != "fp8_mlp":
            x = t["x"]
            h = _norm64(x, t["norm_weight" if kind == "fp8_attention" else "attn_norm_weight"], LAYER_EPS)
            q, k, v = _split_heads(mat(h, "wqkv"), c["heads"], c["kv_heads"])
            z = x + mat(_causal64(_rope64(q, ROPE_THETA), _rope64(k, ROPE_THETA), v), "wo")
        if kind == "fp8_attention":
            return {"output0": z}
        h = _norm64(z, t["norm_weight" if kind == "fp8_mlp" else "mlp_norm_weight"], LAYER_EPS)
        return {"output0": z + mat(_silu64(mat(h, "w_gate")) * mat(h, "w_up"), "w_down")}
    q, k, v = _split_heads(t["x"] @ t["qkv_weight"], c["heads"], c["kv_heads"])
    q, k = _norm64(q, t["q_norm_weight"], EPS), _norm64(k, t["k_norm_weight"], EPS)
    ck, cv = t["cache_k"], t["cache_v"]
    if kind == "qwen3_prefill":
        S = c["seq"]
        q, k = _rope64(q, float(QWEN_ROPE_BASE)), _rope64(k, float(QWEN_ROPE_BASE))
        ck[:, :S], cv[:, :S] = k, v
        o = _causal64(q, k, v)
    else:
        at, half = torch.tensor([float(c["pos"])], dtype=torch.float64, device=q.device), HEAD_DIM // 2
        q, k = (_rope64_at(x, at, float(QWEN_ROPE_BASE), half) for x in (q, k))
        ck[:, c["pos"]], cv[:, c["pos"]] = k[:, 0], v[:, 0]
        rep, o = c["heads"] // c["kv_heads"], torch.empty_like(q)
        for b in range(c["batch"]):
            for g in range(c["kv_heads"]):
                kk, vv = ck[b, :c["pos"] + 1, g].contiguous(), cv[b, :c["pos"] + 1, g].contiguous()
                s = (q[b, 0, g * rep:(g + 1) * rep] @ kk.T.contiguous()) / math.sqrt(HEAD_DIM)
                o[b, 0, g * rep:(g + 1) * rep] = torch.softmax(s, -1) @ vv
        o = o.reshape(c["batch"], 1, -1)
    return {"cache_k": ck, "cache_v": cv, "output0": o @ t["o_weight"]}
