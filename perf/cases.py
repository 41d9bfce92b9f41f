"""Performance cases: what programs built on this library have it compute.

Seven kinds of work, each through the typed launch surface of
``fe2o3_amd.kernels`` on ``fe2o3_amd.runtime`` device buffers, from decoding a
handful of tokens to the largest prefill and offline shapes:

  bf16_linear  C = A B^T on bf16 activations and weights
  fp8_linear   f32 activations quantized with amax scaling, then the e4m3 GEMM
               against weights quantized once
  general      C = alpha A B + beta C on strided bf16 operands, f32 C
  scalar       the sequential f32 GEMM
  flash        attention forward, causal or not, with its log-sum-exp
  softmax      row softmax, with and without a mask
  moe          top-2 router and expert FFN, one layer

``prepare`` lays out what such a program holds before the call (inputs,
weights, outputs, workspaces, prepared launches) and ``run`` enqueues one pass.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from fe2o3_amd import kernels
from fe2o3_amd.runtime import DeviceBuffer, GpuContext

HEAD_DIM = 128
UNBOUNDED = 0xFFFFFFFF  # router capacity

# torch types as the buffers hold them: numpy element type, type of the view
_BF16 = (np.uint16, "<i2", torch.bfloat16)
_F32 = (np.float32, "<f4", torch.float32)
_U8 = (np.uint8, "|u1", torch.uint8)
_U32 = (np.uint32, "<i4", torch.int32)


# ---- cases ------------------------------------------------------------------------------

def listed():
    return [
        # a decoding step's projection: sixteen sequences, one token each
        dict(name="bf16_linear_decode", kind="bf16_linear", m=16, n=4096, k=4096),
        # the headline bf16 GEMM, a prefill projection of 4096 tokens
        dict(name="bf16_linear_4096", kind="bf16_linear", m=4096, n=4096, k=4096),
        # a decoding step of the quantized path, activations quantized on the way
        dict(name="fp8_linear_decode", kind="fp8_linear", m=32, n=8192, k=8192),
        # the quantized path at its headline size
        dict(name="fp8_linear_8192", kind="fp8_linear", m=8192, n=8192, k=8192),
        # a GEMM on windows of larger matrices: nothing aligned, nothing a multiple of a tile
        dict(name="general_ragged", kind="general", m=1000, n=1500, k=700,
             lda=703, ldb=1505, ldc=1507, alpha=1.25, beta=0.5),
        # the smallest configuration, bound by launch and latency
        dict(name="scalar_256", kind="scalar", m=256, n=256, k=256),
        # one prompt of odd length
        dict(name="flash_prompt", kind="flash", batch=1, heads=32, seq=1000, causal=True),
        # the headline attention forward
        dict(name="flash_4096", kind="flash", batch=8, heads=32, seq=4096, causal=False),
        # padded batches: a byte mask over rows that are no multiple of a wave's loads
        dict(name="softmax_masked", kind="softmax", rows=32768, cols=1000, masked=True),
        # long plain rows, bound by memory
        dict(name="softmax_4096", kind="softmax", rows=65536, cols=4096, masked=False),
        # a decoding step through one mixture-of-experts layer
        dict(name="moe_decode", kind="moe", tokens=32, hidden=4096, ffn=14336, experts=8),
        # the headline layer: a prefill of 4096 tokens
        dict(name="moe_4096", kind="moe", tokens=4096, hidden=4096, ffn=14336, experts=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, of):
    """Log-uniform in [lo, hi]; a multiple of `of` in three draws of four."""
    v = _log_int(rng, lo, hi)
    return max(of, v // of * of) if rng.random() < 0.75 else v


def draw(rng):
    kind = rng.choice(["bf16_linear", "fp8_linear", "general", "scalar", "flash", "softmax",
                       "moe"])
    if kind == "bf16_linear":
        return dict(kind=kind, m=_log_int(rng, 1, 4096), n=_multiple(rng, 512, 8192, 64),
                    k=_multiple(rng, 512, 8192, 64))
    if kind == "fp8_linear":
        return dict(kind=kind, m=_log_int(rng, 1, 8192), n=_multiple(rng, 1024, 8192, 64),
                    k=_multiple(rng, 1024, 8192, 64))
    if kind == "general":
        m, n, k = (_log_int(rng, 16, 2048) for _ in range(3))
        pad = rng.choice([0, 0, 8, 5])
        if rng.random() < 0.5:
            m, n, k = (max(16, v // 16 * 16) for v in (m, n, k))
        return dict(kind=kind, m=m, n=n, k=k, lda=k + pad, ldb=n + pad, ldc=n + pad,
                    alpha=round(rng.uniform(0.5, 2.0), 3),
                    beta=rng.choice([0.0, 0.5, 0.25]))
    if kind == "scalar":
        return dict(kind=kind, m=_log_int(rng, 16, 512), n=_log_int(rng, 16, 512),
                    k=_log_int(rng, 16, 512))
    if kind == "flash":
        seq = _multiple(rng, 64, 4096, 64)
        return dict(kind=kind, batch=rng.choice([1, 2, 4, 8]), heads=rng.choice([8, 16, 32]),
                    seq=seq, causal=rng.random() < 0.5)
    if kind == "softmax":
        cols = _multiple(rng, 64, 8192, 64)
        rows = _log_int(rng, 64, min(131072, (1 << 28) // cols))
        return dict(kind=kind, rows=rows, cols=cols, masked=rng.random() < 0.5)
    experts = rng.choice([4, 8, 8, 16])
    return dict(kind="moe", tokens=_log_int(rng, 1, 4096),
                hidden=rng.choice([1024, 2048, 4096]),
                ffn=128 * _log_int(rng, 8, 112 * 8 // max(8, experts)), experts=experts)


# ---- inputs -----------------------------------------------------------------------------

def _generator(seed, part):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + part)


def _normal(shape, std, seed, part, dtype):
    g = _generator(seed, part)
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _inputs(case, seed):
    """The inputs of a case, as torch tensors made from the seed alone."""
    kind = case["kind"]
    if kind == "bf16_linear":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(a=_normal((m, k), 1.0, seed, 0, torch.bfloat16),
                    b=_normal((n, k), k ** -0.5, seed, 1, torch.bfloat16))
    if kind == "fp8_linear":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(x=_normal((m, k), 1.0, seed, 0, torch.float32),
                    w=_normal((n, k), k ** -0.5, seed, 1, torch.float32))
    if kind == "general":
        return dict(a=_normal((case["m"], case["lda"]), 1.0, seed, 0, torch.bfloat16),
                    b=_normal((case["k"], case["ldb"]), case["k"] ** -0.5, seed, 1,
                              torch.bfloat16),
                    c=_normal((case["m"], case["ldc"]), 1.0, seed, 2, torch.float32))
    if kind == "scalar":
        g = _generator(seed, 0)
        m, n, k = case["m"], case["n"], case["k"]
        ab = torch.rand(m * k + k * n, generator=g, device="cuda") * 2 - 1
        return dict(a=ab[:m * k].reshape(m, k), b=ab[m * k:].reshape(k, n))
    if kind == "flash":
        shape = (case["batch"], case["heads"], case["seq"], HEAD_DIM)
        return {t: _normal(shape, 1.0, seed, i, torch.bfloat16) for i, t in enumerate("qkv")}
    if kind == "softmax":
        rows, cols = case["rows"], case["cols"]
        out = dict(x=_normal((rows, cols), 3.0, seed, 0, torch.float32))
        if case["masked"]:  # a padded batch: each row active up to a length of its own
            length = torch.randint(cols // 2, cols + 1, (rows, 1), generator=_generator(seed, 1),
                                   device="cuda")
            out["mask"] = (torch.arange(cols, device="cuda") < length).to(torch.uint8)
        return out
    t, h, f, e = case["tokens"], case["hidden"], case["ffn"], case["experts"]
    return dict(x=_normal((t, h), 1.0, seed, 0, torch.bfloat16),
                logits=_normal((t, e), 1.0, seed, 1, torch.bfloat16),
                w_gate=_normal((e, f, h), 0.02, seed, 2, torch.bfloat16),
                w_up=_normal((e, f, h), 0.02, seed, 3, torch.bfloat16),
                w_down=_normal((e, h, f), 0.02, seed, 4, torch.bfloat16))


# ---- framework buffers and their torch views ----------------------------------------------

class _Span:
    """A device buffer as an array for torch to look at; the view keeps it."""

    def __init__(self, buf: DeviceBuffer, typestr: str):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (buf.count,), "typestr": typestr,
                                         "data": (buf.ptr, False), "version": 3}


def _buffer(shape, kind):
    """A device buffer of `shape` and a torch tensor over its memory."""
    numpy_type, typestr, torch_type = kind
    buf = GpuContext.current().alloc(math.prod(shape), numpy_type)
    return buf, torch.as_tensor(_Span(buf, typestr), device="cuda").view(torch_type).view(shape)


def _holding(t):
    kind = {torch.bfloat16: _BF16, torch.float32: _F32, torch.uint8: _U8}[t.dtype]
    buf, view = _buffer(tuple(t.shape), kind)
    view.copy_(t)
    return buf


def prepare(case, seed):
    kind, ctx, inputs = case["kind"], GpuContext.current(), _inputs(case, seed)
    if kind == "bf16_linear":
        m, n, k = case["m"], case["n"], case["k"]
        c, c_view = _buffer((m, n), _BF16)
        launch = kernels.gemm_bf16_nt_gpu.Kernel.load(ctx).prepare(
            _holding(inputs["a"]), _holding(inputs["b"]), c, m, n, k)
        return dict(kind=kind, launch=launch, out=c_view)
    if kind == "fp8_linear":
        m, n, k = case["m"], case["n"], case["k"]
        w = _holding(inputs["w"])
        state = dict(kind=kind, m=m, n=n, k=k, x=_holding(inputs["x"]))
        for name, shape, t in (("amax", (1,), _F32), ("scale", (1,), _F32),
                               ("w_scale", (1,), _F32), ("codes", (m, k), _U8),
                               ("w_codes", (n, k), _U8), ("out", (m, n), _BF16)):
            state[name], state[name + "_view"] = _buffer(shape, t)
        kernels.amax_f32(w, state["amax"], sync=False)
        kernels.fp8_scale_from_amax(state["amax"], state["w_scale"], sync=False)
        kernels.quantize_e4m3(w, state["w_scale"], state["w_codes"])
        return state
    if kind == "general":
        c, c_view = _buffer((case["m"], case["ldc"]), _F32)
        c_view.copy_(inputs["c"])
        launch = kernels.tiled_gemm_general_v1_gpu.Kernel.load(ctx).prepare(
            _holding(inputs["a"]), _holding(inputs["b"]), c,
            *(case[v] for v in ("m", "n", "k", "lda", "ldb", "ldc", "alpha", "beta")))
        return dict(kind=kind, launch=launch, out=c_view[:, :case["n"]])
    if kind == "scalar":
        c, c_view = _buffer((case["m"], case["n"]), _F32)
        launch = kernels.scalar_gemm_v1_gpu.Kernel.load(ctx).prepare(
            _holding(inputs["a"]), _holding(inputs["b"]), c, case["m"], case["n"], case["k"])
        return dict(kind=kind, launch=launch, out=c_view)
    if kind == "flash":
        b, h, s = case["batch"], case["heads"], case["seq"]
        o, o_view = _buffer((b, h, s, HEAD_DIM), _BF16)
        lse, lse_view = _buffer((b, h, s), _F32)
        launch = kernels.flash_attention_fwd_gpu.Kernel.load(ctx).prepare(
            *(_holding(inputs[t]) for t in "qkv"), o, lse, b, h, s, HEAD_DIM,
            int(case["causal"]), HEAD_DIM ** -0.5)
        return dict(kind=kind, launch=launch, out=dict(o=o_view, lse=lse_view))
    if kind == "softmax":
        y, y_view = _buffer((case["rows"], case["cols"]), _F32)
        mask = _holding(inputs["mask"]) if case["masked"] else None
        launch = kernels.row_softmax_gpu.Kernel.load(ctx).prepare(
            _holding(inputs["x"]), y, mask, case["rows"], case["cols"])
        return dict(kind=kind, launch=launch, out=y_view)
    t, h, f, e = case["tokens"], case["hidden"], case["ffn"], case["experts"]
    routing, views = {}, {}
    for name, count in (("top2", 2 * t), ("requested", e), ("admitted", e), ("offsets", e + 1),
                        ("slots", 2 * t), ("permutation", 2 * t), ("inverse", 2 * t)):
        routing[name], views[name] = _buffer((count,), _U32)
    routing["weights"], views["weights"] = _buffer((2 * t,), _F32)
    out, views["out"] = _buffer((t, h), _BF16)
    workspace = ctx.alloc(kernels.moe_ffn_workspace_bytes(t, h, f, e), np.uint8)
    held = {name: _holding(v) for name, v in inputs.items()}
    return dict(kind=kind, routing=routing, views=views, out=out, workspace=workspace,
                tokens=t, hidden=h, ffn=f, experts=e, **held)


def run(state):
    kind = state["kind"]
    if kind == "fp8_linear":
        kernels.amax_f32(state["x"], state["amax"], sync=False)
        kernels.fp8_scale_from_amax(state["amax"], state["scale"], sync=False)
        kernels.quantize_e4m3(state["x"], state["scale"], state["codes"], sync=False)
        kernels.gemm_fp8_nt(state["codes"], state["w_codes"], state["scale"], state["w_scale"],
                            state["out"], state["m"], state["n"], state["k"], sync=False)
        return dict(codes=state["codes_view"], scale=state["scale_view"], out=state["out_view"])
    if kind == "moe":
        t, h, f, e = (state[v] for v in ("tokens", "hidden", "ffn", "experts"))
        kernels.moe_top2_route(state["logits"], state["routing"], t, e, UNBOUNDED, sync=False)
        kernels.moe_ffn_top2(state["x"], state["w_gate"], state["w_up"], state["w_down"],
                             state["routing"], state["out"], state["workspace"], t, h, f, e,
                             sync=False)
        return state["views"]
    state["launch"].launch_async()
    return state["out"]


# ---- what a pass cannot do without, and what it may differ by ------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("bf16_linear", "fp8_linear", "general", "scalar"):
        m, n, k = case["m"], case["n"], case["k"]
        moved = {"bf16_linear": 2 * (m * k + n * k + m * n),
                 "fp8_linear": 4 * m * k + m * k + n * k + 2 * m * n,
                 "general": 2 * (m * k + k * n) + 8 * m * n,
                 "scalar": 4 * (m * k + k * n + m * n)}[kind]
        return dict(bytes=moved, flops=2 * m * n * k)
    if kind == "flash":
        rows = case["batch"] * case["heads"] * case["seq"]
        flops = 4 * rows * case["seq"] * HEAD_DIM
        return dict(bytes=rows * (4 * HEAD_DIM * 2 + 4),
                    flops=flops // 2 if case["causal"] else flops)
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return dict(bytes=n * (9 if case["masked"] else 8), flops=5 * n)
    t, h, f, e = case["tokens"], case["hidden"], case["ffn"], case["experts"]
    used = min(e, 2 * t)  # experts whose weights are read
    return dict(bytes=2 * (3 * used * f * h + 2 * t * h + t * e) + 4 * (10 * t + 3 * e),
                flops=2 * 2 * t * 3 * f * h)


def tolerance(case):
    kind = case["kind"]
    if kind == "scalar":
        return "exact"  # the sequential unfused sum is the contract
    if kind == "softmax":
        return dict(rel=5e-7)  # f32 sums in another order, exp to an ulp: 8e-8 against 64 bits
    if kind == "general":
        return dict(rel=1e-6)  # f32 sums of exact products in another order: 1.4e-7 at k = 700
    # one bf16 rounding of each output (1.7e-3 against 64 bits), and one of what the second
    # product reads in attention and the expert FFN (2.3e-3)
    return dict(rel=6e-3 if kind.endswith("linear") else 8e-3)


# ---- the same results in 64 bits -----------------------------------------------------------

def _e4m3(x):
    """Codes and f32 scale of the amax quantization."""
    scale = x.abs().max().clamp_min(torch.finfo(torch.float32).tiny) / 448.0
    return (x / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), scale


def _exact_flash(case, inputs):
    s = case["seq"]
    q, k, v = (inputs[t].reshape(-1, s, HEAD_DIM) for t in "qkv")
    o = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    lse = torch.empty(q.shape[:2], dtype=torch.float64, device="cuda")
    future = torch.ones(s, s, dtype=torch.bool, device="cuda").triu(1)
    for i in range(q.shape[0]):
        score = (q[i].double() @ k[i].double().t().contiguous()) * HEAD_DIM ** -0.5
        if case["causal"]:
            score.masked_fill_(future, -math.inf)
        lse[i] = torch.logsumexp(score, dim=1)
        o[i] = torch.exp(score - lse[i][:, None]) @ v[i].double()
    shape = (case["batch"], case["heads"], s)
    return dict(o=o.view(*shape, HEAD_DIM), lse=lse.view(shape))


def _exact_moe(case, inputs):
    t, h, e = case["tokens"], case["hidden"], case["experts"]
    logits = inputs["logits"].double()
    score, top2 = torch.sort(logits, dim=1, descending=True, stable=True)
    score, top2 = score[:, :2], top2[:, :2]
    w0 = torch.sigmoid(score[:, 0] - score[:, 1])
    weights = torch.stack([w0, 1.0 - w0], dim=1)
    out = torch.zeros(t, h, dtype=torch.float64, device="cuda")
    for x in range(e):
        token, rank = torch.where(top2 == x)
        if token.numel() == 0:
            continue
        rows = inputs["x"][token].double()
        gate = rows @ inputs["w_gate"][x].double().t().contiguous()
        up = rows @ inputs["w_up"][x].double().t().contiguous()
        y = (gate * torch.sigmoid(gate) * up) @ inputs["w_down"][x].double().t().contiguous()
        out.index_add_(0, token, y * weights[token, rank][:, None])
    none = {name: None for name in ("top2", "requested", "admitted", "offsets", "slots",
                                    "permutation", "inverse")}
    return dict(weights=weights.reshape(-1), out=out, **none)


def exact(case, seed):
    kind, inputs = case["kind"], _inputs(case, seed)
    if kind == "bf16_linear":
        return inputs["a"].double() @ inputs["b"].double().t().contiguous()
    if kind == "fp8_linear":
        (x, sx), (w, sw) = _e4m3(inputs["x"]), _e4m3(inputs["w"])
        out = x.double() @ w.double().t().contiguous()
        return dict(codes=None, scale=sx.double().view(1), out=out * (sx.double() * sw.double()))
    if kind == "general":
        n, k = case["n"], case["k"]
        ab = inputs["a"][:, :k].double() @ inputs["b"][:, :n].double()
        return case["alpha"] * ab + case["beta"] * inputs["c"][:, :n].double()
    if kind == "scalar":
        return inputs["a"].double() @ inputs["b"].double()
    if kind == "flash":
        return _exact_flash(case, inputs)
    if kind == "softmax":
        x = inputs["x"].double()
        if case["masked"]:
            x.masked_fill_(inputs["mask"] == 0, -math.inf)
        return torch.softmax(x, dim=1)
    return _exact_moe(case, inputs)
