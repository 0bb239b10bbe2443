"""The work that programs built on this package have it do, case by case.

A case is a dict of plain values.  Its "kind" names the entry point:

* scan     selective_scan_fn, forward and backward (training through the scan);
* block    MambaSimple, forward and backward (one layer of a training step);
* prefill  MambaSimple over a whole prompt without autograd, filling the decode cache;
* step     MambaSimple.step_prenorm, one token of a layer, launched from Python;
* decode   CausalLM one token at a time through GraphedStep;
* norm     residual add + RMSNorm, forward and backward;
* conv     causal depthwise conv1d + SiLU, forward and backward.

Inputs, weights and caches come from the seed alone.  ``exact`` restates each
computation in float64 with plain torch, from the same rounded inputs.
"""
import math

import torch
import torch.nn.functional as F

from mamba_amd.models import CausalLM, CausalLMConfig
from mamba_amd.models.causal_lm import GraphedStep
from mamba_amd.modules import MambaSimple, RMSNorm
from mamba_amd.ops.causal_conv1d import causal_conv1d_fn
from mamba_amd.ops.rms_norm import rms_norm_fn
from mamba_amd.ops.selective_scan_interface import selective_scan_fn

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
CONV = 4          # the models' conv width


# ---------------------------------------------------------------- cases --
def listed():
    return [
        # a unit-test-size scan: latency and launches only
        {"name": "scan_small", "kind": "scan", "batch": 2, "dim": 64, "state": 16, "len": 256, "dtype": "f32"},
        # the scan of a 768-wide model's training step in fp32
        {"name": "scan_train", "kind": "scan", "batch": 8, "dim": 1536, "state": 16, "len": 2048, "dtype": "f32"},
        # the scan of a 2560-wide model on long sequences with bf16 activations
        {"name": "scan_long", "kind": "scan", "batch": 4, "dim": 5120, "state": 16, "len": 8192, "dtype": "bf16"},
        # next-token training cuts sequences to one short of the context: every row starts off its alignment
        {"name": "scan_ragged", "kind": "scan", "batch": 8, "dim": 1536, "state": 16, "len": 2047, "dtype": "f32"},
        # a small-state model of a width that is no multiple of 16 (500, expanded twice)
        {"name": "scan_odd_width", "kind": "scan", "batch": 8, "dim": 1000, "state": 8, "len": 2048, "dtype": "f32"},
        # a large-state model
        {"name": "scan_wide_state", "kind": "scan", "batch": 4, "dim": 1536, "state": 64, "len": 1024,
         "dtype": "bf16"},
        # one layer of a 1024-wide model's training step
        {"name": "block_train", "kind": "block", "batch": 8, "len": 2048, "width": 1024, "state": 16,
         "dtype": "bf16"},
        # one layer of a long prompt's prefill
        {"name": "block_prefill", "kind": "prefill", "batch": 1, "len": 32768, "width": 768, "state": 16,
         "dtype": "bf16"},
        # one layer of a decode step called from Python
        {"name": "block_step", "kind": "step", "batch": 16, "width": 768, "state": 16, "dtype": "bf16"},
        # a token of a 24-layer model, replayed as one graph
        {"name": "lm_decode", "kind": "decode", "batch": 16, "width": 768, "layers": 24, "vocab": 50280,
         "state": 16, "dtype": "bf16"},
        # the norm in front of every block, with the residual stream
        {"name": "norm_train", "kind": "norm", "rows": 32768, "width": 768, "dtype": "bf16"},
        # the conv of a training step on sequences one short of the context
        {"name": "conv_train", "kind": "conv", "batch": 8, "dim": 1536, "len": 2047, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(rng, v, unit):
    """v itself, or v rounded to the unit (half of the draws each)."""
    return v if rng.random() < 0.5 else max(unit, unit * round(v / unit))


def draw(rng):
    kind = rng.choice(["scan"] * 6 + ["block"] * 2 + ["prefill", "step", "decode", "norm", "conv"])
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    if kind == "scan":
        while True:
            c = {"kind": kind, "batch": _log(rng, 1, 16), "dim": _near(rng, _log(rng, 48, 5120), 16),
                 "state": rng.choice([16, 16, 16, 16, 4, 8, 24, 32, 64]), "len": _near(rng, _log(rng, 100, 8192), 64),
                 "dtype": dtype}
            if c["batch"] * c["dim"] * c["len"] * max(16, c["state"]) <= 4 * 5120 * 8192 * 16 // 8:
                return c
    if kind == "block":
        while True:
            c = {"kind": kind, "batch": _log(rng, 1, 16), "len": _near(rng, _log(rng, 100, 8192), 64),
                 "width": _near(rng, _log(rng, 128, 1536), 64), "state": rng.choice([16, 16, 16, 8, 32]),
                 "dtype": dtype}
            if c["batch"] * c["len"] * c["width"] <= 8 * 2048 * 768 // 2:
                return c
    if kind == "prefill":
        return {"kind": kind, "batch": _log(rng, 1, 2), "len": _near(rng, _log(rng, 512, 16384), 64),
                "width": _near(rng, _log(rng, 256, 1024), 64), "state": 16, "dtype": rng.choice(["bf16", "f16"])}
    if kind == "step":
        return {"kind": kind, "batch": _log(rng, 1, 64), "width": _near(rng, _log(rng, 128, 2048), 64),
                "state": rng.choice([16, 16, 8, 32]), "dtype": rng.choice(["bf16", "f16"])}
    if kind == "decode":
        return {"kind": kind, "batch": _log(rng, 1, 64), "width": 64 * rng.randint(4, 12), "layers": rng.randint(2, 24),
                "vocab": rng.choice([32000, 50280]), "state": 16, "dtype": "bf16"}
    if kind == "norm":
        return {"kind": kind, "rows": _log(rng, 16, 32768), "width": _near(rng, _log(rng, 128, 2560), 64),
                "dtype": dtype}
    return {"kind": kind, "batch": _log(rng, 1, 8), "dim": _near(rng, _log(rng, 128, 3072), 16),
            "len": _near(rng, _log(rng, 64, 4096), 64), "dtype": dtype}


# --------------------------------------------------------------- inputs --
class _Draw:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.gen, device="cuda") * scale).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return (torch.rand(*shape, generator=self.gen, device="cuda") * (hi - lo) + lo).to(dtype)


def _delta_bias(d, dim):
    # softplus(bias) log-uniform in [0.001, 0.1], the models' initialisation
    dt = torch.exp(d.uniform(dim, lo=math.log(1e-3), hi=math.log(0.1)))
    return dt + torch.log(-torch.expm1(-dt))


def _log_A(dim, state):
    return torch.log(torch.arange(1, state + 1, device="cuda", dtype=torch.float32)).repeat(dim, 1)


def _scan_inputs(case, seed):
    d, dt = _Draw(seed), DT[case["dtype"]]
    b, n, l, dim = case["batch"], case["state"], case["len"], case["dim"]
    return {
        "u": d.normal(b, dim, l, dtype=dt), "delta": d.normal(b, dim, l, scale=0.5, dtype=dt),
        "A": -torch.exp(_log_A(dim, n) + d.normal(dim, n, scale=0.05)),
        "B": d.normal(b, 1, n, l, dtype=dt), "C": d.normal(b, 1, n, l, dtype=dt),
        "D": 1.0 + d.normal(dim, scale=0.1), "z": d.normal(b, dim, l, dtype=dt),
        "delta_bias": _delta_bias(d, dim),
    }, d.normal(b, dim, l, dtype=dt)


def _block_weights(d, width, state, dt, prefix=""):
    inner, rank = 2 * width, math.ceil(width / 16)
    w = {
        "input_proj.weight": d.uniform(2 * inner, width, lo=-1, hi=1, dtype=dt) * width ** -0.5,
        "short_conv.weight": d.uniform(inner, 1, CONV, lo=-0.5, hi=0.5, dtype=dt),
        "ssm_param_proj.weight": d.uniform(rank + 2 * state, inner, lo=-1, hi=1, dtype=dt) * inner ** -0.5,
        "delta_proj.weight": d.uniform(inner, rank, lo=-1, hi=1, dtype=dt) * rank ** -0.5,
        "delta_proj.bias": _delta_bias(d, inner).to(dt),
        "log_A": _log_A(inner, state), "D": 1.0 + d.normal(inner, scale=0.1),
        "output_proj.weight": d.uniform(width, inner, lo=-1, hi=1, dtype=dt) * inner ** -0.5,
    }
    return {prefix + k: v for k, v in w.items()}


def _cache(d, batch, width, state, dt):
    # of a sequence's size after some tokens: conv inputs of order one, a state of a few tenths
    return (d.normal(batch, 2 * width, CONV, dtype=dt), d.normal(batch, 2 * width, state, scale=0.3))


def _block_inputs(case, seed):
    d, dt = _Draw(seed), DT[case["dtype"]]
    w = _block_weights(d, case["width"], case["state"], dt)
    x = d.normal(case["batch"], case["len"], case["width"], dtype=dt)
    return w, x, d.normal(case["batch"], case["len"], case["width"], dtype=dt)


def _step_inputs(case, seed):
    d, dt = _Draw(seed), DT[case["dtype"]]
    b, width = case["batch"], case["width"]
    w = _block_weights(d, width, case["state"], dt)
    norm = d.normal(width, scale=0.1, dtype=dt)
    x, res = d.normal(b, width, dtype=dt), d.normal(b, width, dtype=dt)
    return w, norm, x, res, _cache(d, b, width, case["state"], dt)


def _lm_inputs(case, seed):
    d, dt = _Draw(seed), DT[case["dtype"]]
    w = {"embedding.weight": d.normal(case["vocab"], case["width"], scale=0.02, dtype=dt)}
    for i in range(case["layers"]):
        w["layers.%d.norm.weight" % i] = d.normal(case["width"], scale=0.1, dtype=dt)
        w.update(_block_weights(d, case["width"], case["state"], dt, "layers.%d.mamba." % i))
    w["norm.weight"] = d.normal(case["width"], scale=0.1, dtype=dt)
    w["lm_head.weight"] = w["embedding.weight"]
    caches = [_cache(d, case["batch"], case["width"], case["state"], dt) for _ in range(case["layers"])]
    ids = torch.randint(case["vocab"], (case["batch"],), generator=d.gen, device="cuda")
    return w, caches, ids


def _norm_inputs(case, seed):
    d, dt = _Draw(seed), DT[case["dtype"]]
    shape = (case["rows"], case["width"])
    return (d.normal(*shape, dtype=dt), d.normal(case["width"], scale=0.1, dtype=dt), d.normal(*shape, dtype=dt),
            d.normal(*shape, dtype=dt), d.normal(*shape, dtype=dt))


def _conv_inputs(case, seed):
    d, dt = _Draw(seed), DT[case["dtype"]]
    b, dim, l = case["batch"], case["dim"], case["len"]
    return (d.normal(b, dim, l, dtype=dt), d.uniform(dim, 1, CONV, lo=-0.5, hi=0.5, dtype=dt),
            d.uniform(dim, lo=-0.5, hi=0.5, dtype=dt), d.normal(b, dim, l, dtype=dt))


def _mamba(case, weights, dt):
    m = MambaSimple(case["width"], state_dim=case["state"], conv_kernel=CONV, device="cuda", dtype=dt)
    m.load_state_dict(weights)
    return m


def prepare(case, seed):
    kind, dt = case["kind"], DT[case["dtype"]]
    if kind == "scan":
        x, dout = _scan_inputs(case, seed)
        return {"kind": kind, "x": {k: v.requires_grad_(True) for k, v in x.items()}, "dout": dout}
    if kind == "block":
        w, x, dout = _block_inputs(case, seed)
        return {"kind": kind, "block": _mamba(case, w, dt), "x": x.requires_grad_(True), "dout": dout}
    if kind == "prefill":
        w, x, _ = _block_inputs(case, seed)
        m = _mamba(case, w, dt)
        return {"kind": kind, "block": m, "x": x, "cache": m.allocate_inference_cache(case["batch"])}
    if kind == "step":
        w, nw, x, res, cache = _step_inputs(case, seed)
        norm = RMSNorm(case["width"], device="cuda", dtype=dt)
        norm.load_state_dict({"weight": nw})
        return {"kind": kind, "block": _mamba(case, w, dt), "norm": norm, "x": x, "residual": res, "cache": cache}
    if kind == "decode":
        w, caches, ids = _lm_inputs(case, seed)
        cfg = CausalLMConfig(vocab_size=case["vocab"], model_dim=case["width"], state_dim=case["state"],
                             conv_kernel=CONV, num_layers=case["layers"])
        lm = CausalLM(cfg, device="cuda", dtype=dt).eval()
        lm.load_state_dict(w)
        return {"kind": kind, "step": GraphedStep(lm, caches, case["batch"]), "lm": lm, "cache": caches, "ids": ids}
    if kind == "norm":
        x, w, res, dout, ds = _norm_inputs(case, seed)
        return {"kind": kind, "in": [t.requires_grad_(True) for t in (x, w, res)], "douts": (dout, ds)}
    x, w, b, dout = _conv_inputs(case, seed)
    return {"kind": kind, "in": [t.requires_grad_(True) for t in (x, w, b)], "dout": dout}


# ----------------------------------------------------------------- pass --
def run(s):
    kind = s["kind"]
    if kind == "scan":
        x = s["x"]
        out = selective_scan_fn(x["u"], x["delta"], x["A"], x["B"], x["C"], x["D"], z=x["z"],
                                delta_bias=x["delta_bias"], delta_softplus=True)
        return {"out": out.detach(), **dict(zip(x, torch.autograd.grad(out, list(x.values()), s["dout"])))}
    if kind == "block":
        out = s["block"](s["x"])
        names, params = zip(*s["block"].named_parameters())
        grads = torch.autograd.grad(out, [s["x"], *params], s["dout"])
        return {"out": out.detach(), **dict(zip(("x",) + names, grads))}
    if kind == "prefill":
        with torch.no_grad():
            out = s["block"](s["x"], inference_cache=s["cache"])
        return {"out": out, "conv_state": s["cache"][0], "ssm_state": s["cache"][1]}
    if kind == "step":
        with torch.no_grad():
            out, res = s["block"].step_prenorm(s["x"], s["residual"], s["norm"], *s["cache"])
        return {"out": out, "residual": res, "conv_state": s["cache"][0], "ssm_state": s["cache"][1]}
    if kind == "decode":
        logits = s["step"](s["ids"])
        return {"logits": logits, "conv_state": [c for c, _ in s["cache"]], "ssm_state": [h for _, h in s["cache"]]}
    if kind == "norm":
        x, w, res = s["in"]
        out, stream = rms_norm_fn(x, w, res, prenorm=True)
        dx, dw, dres = torch.autograd.grad((out, stream), (x, w, res), s["douts"])
        return {"out": out.detach(), "stream": stream.detach(), "dx": dx, "dw": dw, "dres": dres}
    x, w, b = s["in"]
    out = causal_conv1d_fn(x, w, b, "silu")
    dx, dw, db = torch.autograd.grad(out, (x, w, b), s["dout"])
    return {"out": out.detach(), "dx": dx, "dw": dw, "db": db}


# ----------------------------------------------------------------- work --
def _block_sizes(case):
    width, n = case["width"], case["state"]
    inner, rank = 2 * width, math.ceil(width / 16)
    gemm = 2 * inner * width + (rank + 2 * n) * inner + inner * rank + width * inner    # weights
    return inner, rank, gemm


def work(case):
    kind, es = case["kind"], SIZE[case["dtype"]]
    # per (channel, state, step): forward 1 exp, 2 products, 2 FMAs; backward the same again (the states are
    # recomputed, not kept) without the output's FMA, and 9 more products and sums
    fwd, bwd = 7, 17
    if kind == "scan":
        b, dim, n, l = case["batch"], case["dim"], case["state"], case["len"]
        el, bc, par = b * dim * l, b * n * l, dim * n
        # u, delta, z, out; then u, delta, z, dout, du, ddelta, dz; B and C both ways and their gradients
        return {"bytes": es * (11 * el + 6 * bc) + 4 * (3 * par + 6 * dim), "flops": (fwd + bwd) * el * n}
    if kind in ("block", "prefill"):
        inner, _, gemm = _block_sizes(case)
        rows = case["batch"] * case["len"]
        if kind == "prefill":
            return {"bytes": es * (2 * rows * case["width"] + gemm) + 4 * inner * case["state"] * (case["batch"] + 1),
                    "flops": 2 * rows * gemm + rows * inner * (fwd * case["state"] + 12)}
        return {"bytes": es * (4 * rows * case["width"] + 2 * gemm) + 8 * inner * case["state"],
                "flops": 6 * rows * gemm + rows * inner * ((fwd + bwd) * case["state"] + 36)}
    if kind in ("step", "decode"):
        inner, _, gemm = _block_sizes(case)
        b, n, width = case["batch"], case["state"], case["width"]
        layer = es * (gemm + 2 * b * inner * CONV) + 4 * (2 * b * inner * n + inner * n)
        ops = 2 * b * gemm + b * inner * (fwd * n + 12)
        if kind == "step":
            return {"bytes": layer + es * 4 * b * width, "flops": ops}
        head = case["vocab"] * width
        return {"bytes": case["layers"] * layer + es * (head + b * case["vocab"]),
                "flops": case["layers"] * ops + 2 * b * head}
    if kind == "norm":
        el = case["rows"] * case["width"]
        # x, residual, out, stream; then stream, dout, dstream, dx (dres is dx)
        return {"bytes": es * 8 * el, "flops": 16 * el}
    el = case["batch"] * case["dim"] * case["len"]
    return {"bytes": es * 5 * el, "flops": (4 * CONV + 4 * CONV + 20) * el}


def tolerance(case):
    kind, dt = case["kind"], case["dtype"]
    half = {"bf16": 1e-2, "f16": 2e-3}
    if dt == "f32":
        return {"rel": 1e-5 if kind != "block" else 1e-4}
    return {"rel": half[dt]}


# -------------------------------------------------------------- float64 --
class _Scan64(torch.autograd.Function):
    """The recurrence h_t = exp(delta A) h + delta u B, y_t = C h and its adjoint, float64, time first."""

    PART = 256

    @staticmethod
    def forward(ctx, u, delta, A, B, C):
        # u, delta: (l, b, d); A: (d, n); B, C: (l, b, n)
        l, b, d = u.shape
        h = torch.zeros(b, d, A.shape[1], dtype=torch.float64, device=u.device)
        hs = torch.empty(l, b, d, A.shape[1], dtype=torch.float64, device=u.device)
        y = torch.empty_like(u)
        for t0 in range(0, l, _Scan64.PART):
            p = slice(t0, min(l, t0 + _Scan64.PART))
            a = torch.exp(delta[p, :, :, None] * A)
            v = (delta[p] * u[p])[..., None] * B[p, :, None, :]
            for t in range(a.shape[0]):
                torch.addcmul(v[t], a[t], h, out=hs[t0 + t])
                h = hs[t0 + t]
            y[p] = (hs[p] * C[p, :, None, :]).sum(-1)
        ctx.save_for_backward(u, delta, A, B, C, hs)
        return y, h.clone()

    @staticmethod
    def backward(ctx, dy, _):
        u, delta, A, B, C, hs = ctx.saved_tensors
        l = u.shape[0]
        du, ddelta, dA = torch.empty_like(u), torch.empty_like(u), torch.zeros_like(A)
        dB, dC = torch.empty_like(B), torch.empty_like(C)
        ga = torch.zeros_like(hs[0])
        for t1 in range(l, 0, -_Scan64.PART):
            t0 = max(0, t1 - _Scan64.PART)
            p = slice(t0, t1)
            a = torch.exp(delta[p, :, :, None] * A)
            g = dy[p][..., None] * C[p, :, None, :]
            for t in range(t1 - t0 - 1, -1, -1):
                g[t] += ga
                ga = g[t] * a[t]
            prev = torch.cat([hs[t0 - 1:t0] if t0 else torch.zeros_like(hs[:1]), hs[t0:t1 - 1]])
            gb = (g * B[p, :, None, :]).sum(-1)
            w = g * a * prev
            du[p] = delta[p] * gb
            ddelta[p] = u[p] * gb + (w * A).sum(-1)
            dA += (w * delta[p][..., None]).sum((0, 1))
            dB[p] = (g * (delta[p] * u[p])[..., None]).sum(2)
            dC[p] = (hs[p] * dy[p][..., None]).sum(2)
        return du, ddelta, dA, dB, dC


def _scan64(u, delta, A, B, C, D, z, bias):
    """(b, d, l) u, delta, z; (b, n, l) B, C: the gated scan with softplus, and the last state."""
    dt = F.softplus(delta + bias[:, None])
    first = (u.permute(2, 0, 1).contiguous(), dt.permute(2, 0, 1).contiguous(), A,
             B.permute(2, 0, 1).contiguous(), C.permute(2, 0, 1).contiguous())
    y, h = _Scan64.apply(*first)
    return (y.permute(1, 2, 0) + D[:, None] * u) * F.silu(z), h


def _block64(w, x, width, state):
    """x: (b, l, width); returns (out, xz, last state)."""
    inner, rank = 2 * width, math.ceil(width / 16)
    xz = (x @ w["input_proj.weight"].t()).transpose(1, 2)
    xi, z = xz[:, :inner], xz[:, inner:]
    xc = F.silu(F.conv1d(xi, w["short_conv.weight"], groups=inner, padding=CONV - 1)[..., :x.shape[1]])
    dbl = w["ssm_param_proj.weight"] @ xc
    delta = w["delta_proj.weight"] @ dbl[:, :rank]
    y, h = _scan64(xc, delta, -torch.exp(w["log_A"]), dbl[:, rank:rank + state], dbl[:, rank + state:], w["D"], z,
                   w["delta_proj.bias"])
    return y.transpose(1, 2) @ w["output_proj.weight"].t(), xi, h


def _step64(w, x, conv_state, h, width, state):
    """One token of a block: x (b, width); returns (out, conv_state, h)."""
    inner, rank = 2 * width, math.ceil(width / 16)
    xz = x @ w["input_proj.weight"].t()
    conv_state = torch.cat([conv_state[..., 1:], xz[:, :inner, None]], -1)
    xc = F.silu((conv_state * w["short_conv.weight"][:, 0]).sum(-1))
    dbl = xc @ w["ssm_param_proj.weight"].t()
    dt = F.softplus(dbl[:, :rank] @ w["delta_proj.weight"].t() + w["delta_proj.bias"])
    B, C = dbl[:, rank:rank + state], dbl[:, rank + state:]
    h = torch.exp(dt[..., None] * -torch.exp(w["log_A"])) * h + (dt * xc)[..., None] * B[:, None]
    y = ((h * C[:, None]).sum(-1) + w["D"] * xc) * F.silu(xz[:, inner:])
    return y @ w["output_proj.weight"].t(), conv_state, h


def _norm64(x, w, eps=1e-6):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * (1 + w)


def _conv_norm64(tensors):
    return [t.detach().double().requires_grad_(True) for t in tensors]


def exact(case, seed):
    kind = case["kind"]
    if kind == "scan":
        x, dout = _scan_inputs(case, seed)
        x = {k: v.double().requires_grad_(True) for k, v in x.items()}
        out, _ = _scan64(x["u"], x["delta"], x["A"], x["B"][:, 0], x["C"][:, 0], x["D"], x["z"], x["delta_bias"])
        return {"out": out.detach(), **dict(zip(x, torch.autograd.grad(out, list(x.values()), dout.double())))}
    if kind == "block":
        w, x, dout = _block_inputs(case, seed)
        # in the order of the module's parameters
        order = ["log_A", "D", "input_proj.weight", "short_conv.weight", "ssm_param_proj.weight", "delta_proj.weight",
                 "delta_proj.bias", "output_proj.weight"]
        w = {k: w[k].double().requires_grad_(True) for k in order}
        x = x.double().requires_grad_(True)
        out, _, _ = _block64(w, x, case["width"], case["state"])
        return {"out": out.detach(), **dict(zip(["x", *order], torch.autograd.grad(out, [x, *w.values()], dout.double())))}
    if kind == "prefill":
        w, x, _ = _block_inputs(case, seed)
        with torch.no_grad():
            out, xi, h = _block64({k: v.double() for k, v in w.items()}, x.double(), case["width"], case["state"])
        return {"out": out, "conv_state": F.pad(xi, (CONV, 0))[..., -CONV:].contiguous(), "ssm_state": h}
    if kind == "step":
        w, nw, x, res, (conv, h) = _step_inputs(case, seed)
        w = {k: v.double() for k, v in w.items()}
        stream = x.double() + res.double()
        out, conv, h = _step64(w, _norm64(stream, nw.double()), conv.double(), h.double(), case["width"], case["state"])
        return {"out": out, "residual": stream, "conv_state": conv, "ssm_state": h}
    if kind == "decode":
        w, caches, ids = _lm_inputs(case, seed)
        w = {k: v.double() for k, v in w.items()}
        stream, convs, hs = w["embedding.weight"][ids], [], []
        for i, (conv, h) in enumerate(caches):
            p = "layers.%d.mamba." % i
            layer = {k[len(p):]: v for k, v in w.items() if k.startswith(p)}
            out, conv, h = _step64(layer, _norm64(stream, w["layers.%d.norm.weight" % i]), conv.double(), h.double(),
                                   case["width"], case["state"])
            stream = stream + out
            convs.append(conv)
            hs.append(h)
        return {"logits": _norm64(stream, w["norm.weight"]) @ w["lm_head.weight"].t(), "conv_state": convs,
                "ssm_state": hs}
    if kind == "norm":
        x, w, res, dout, ds = _norm_inputs(case, seed)
        x, w, res = _conv_norm64((x, w, res))
        stream = x + res
        out = _norm64(stream, w)
        dx, dw, dres = torch.autograd.grad((out, stream), (x, w, res), (dout.double(), ds.double()))
        return {"out": out.detach(), "stream": stream.detach(), "dx": dx, "dw": dw, "dres": dres}
    x, w, b, dout = _conv_inputs(case, seed)
    x, w, b = _conv_norm64((x, w, b))
    out = F.silu(F.conv1d(x, w, b, groups=case["dim"], padding=CONV - 1)[..., :case["len"]])
    dx, dw, db = torch.autograd.grad(out, (x, w, b), dout.double())
    return {"out": out.detach(), "dx": dx, "dw": dw, "db": db}
