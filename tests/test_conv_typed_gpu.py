"""The causal conv's parameters in the rows' type or fp32 (mixed types go
through fp32): gradients of the parameters' types against float64 autograd, the
same bits on every run, over widths 1 to 4, row tiles that end inside a vector,
several tiles per row and more (batch row, tile) pairs than a wave has lanes.

Tolerance: the fp32 sums are within 1e-5 of their size; one rounding to the
parameter's type adds half a spacing, at most 2^-8 (bf16, 8 significant bits) or 2^-11
(fp16) of it.
"""
import sys

import pytest
import torch
import torch.nn.functional as F

from mamba_amd.ops.causal_conv1d import causal_conv1d_fn

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
CASES = [(2, 5, 7, 4, BF16, BF16, BF16), (1, 3, 2049, 3, F16, F16, F16), (70, 2, 33, 2, BF16, BF16, None),
         (3, 4, 5000, 4, F32, F32, F32), (2, 6, 65, 1, BF16, F32, F32), (2, 6, 64, 4, F16, F32, F16),
         (2, 3, 100, 4, F32, BF16, BF16)]


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(v).replace("torch.", "") for v in c) for c in CASES])
def test_parameter_types(case):
    b, d, l, width, xt, wt, bt = case
    print(f"\n[conv typed] {case}", flush=True)
    sys.stdout.flush()
    g = torch.Generator().manual_seed(l + width)
    x = torch.randn(b, d, l, generator=g).to(xt).to(DEV).requires_grad_(True)
    w = (torch.rand(d, 1, width, generator=g) - 0.5).to(wt).to(DEV).requires_grad_(True)
    bias = (torch.rand(d, generator=g) - 0.5).to(bt).to(DEV).requires_grad_(True) if bt is not None else None
    dout = torch.randn(b, d, l, generator=g).to(xt).to(DEV)
    ins = [t for t in (x, w, bias) if t is not None]
    got = torch.autograd.grad(causal_conv1d_fn(x, w, bias, "silu"), ins, dout)
    again = torch.autograd.grad(causal_conv1d_fn(x, w, bias, "silu"), ins, dout)
    ref = [t.detach().double().requires_grad_(True) for t in ins]
    out = F.silu(F.conv1d(ref[0], ref[1], ref[2] if bias is not None else None, groups=d, padding=width - 1)[..., :l])
    want = torch.autograd.grad(out, ref, dout.double())
    for t, a, c, r in zip(ins, got, again, want):
        assert a.dtype == t.dtype and a.shape == t.shape and torch.equal(a, c)
        eps = {F32: 0.0, BF16: 2.0 ** -8, F16: 2.0 ** -11}[t.dtype]
        assert (a.double() - r).abs().le((1e-5 + eps) * r.abs() + 1e-5 * r.abs().max()).all()
