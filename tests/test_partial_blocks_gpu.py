"""GPU parity of the partial-block scan kernels: channel blocks that end with
their group (dim or channels per group not a multiple of 16) and fewer than 16
states, forward and backward against the float64 C oracle.

Sizes sit at the edges: one channel, 15 to 17 and 33 of them, groups of 8, 17
and 24 channels, dstate 1, 7, 15 and 16, seqlens around a 16-step chunk, a
64-step super-chunk and a 32-step chunk pair, sequence segments, state slices
(dstate 32) of a ragged dim, constant B / C, and calls without a workspace.
The tolerance is the parity tests' (fp32 1e-3, 16-bit types 2e-2: the rounding
of inputs and outputs, 2^-8 for bf16, over sums of a few hundred terms).
"""
import sys

import pytest
import torch

from mamba_amd import selective_scan as ss
from oracle import c_oracle
from oracle.selective_scan_ref import make_inputs
from tests._util import assert_close

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
TOL = {F32: 1e-3, BF16: 2e-2, F16: 2e-2}

# batch, dim, groups, dstate, seqlen, dtype, var_B, var_C, z, workspace
CASES = [
    (1, 1, 1, 1, 1, F32, True, True, True, "auto"),
    (2, 15, 1, 16, 64, F32, True, True, True, "auto"),
    (2, 17, 1, 16, 65, BF16, True, True, False, "auto"),
    (3, 33, 1, 7, 63, F32, True, True, True, None),
    (2, 32, 1, 15, 96, F16, True, True, True, "auto"),
    (2, 24, 3, 16, 48, F32, True, True, True, None),
    (2, 34, 2, 3, 47, F32, True, True, True, "auto"),
    (2, 72, 3, 16, 200, BF16, True, True, True, "auto"),
    (1, 40, 1, 8, 1500, F32, True, True, True, "auto"),
    (1, 40, 1, 8, 1500, F32, True, True, False, None),
    (2, 24, 1, 8, 100, F32, False, False, True, "auto"),
    (1, 40, 1, 5, 1030, BF16, False, True, True, "auto"),
    (1, 40, 2, 16, 1030, F32, True, False, True, "auto"),
    (2, 20, 1, 32, 130, F32, True, True, True, "auto"),
    (1, 20, 1, 48, 1100, BF16, True, True, True, "auto"),
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(v).replace("torch.", "") for v in c) for c in CASES])
def test_partial_blocks_match_oracle(case):
    b, d, G, n, l, dt, vB, vC, hz, ws = case
    print(f"\n[partial] {case}", flush=True)
    sys.stdout.flush()
    x = make_inputs(b, d, n, l, seed=900 + d + l, dtype=dt, n_groups=G, var_B=vB, var_C=vC, has_z=hz)
    t = {k: v.to(DEV) if v is not None else None for k, v in x.items()}
    # a guard row on either side of x and dA: the lanes without a channel or state write nothing
    nck = ss.n_chunks(l)
    xg = torch.full((b * nck * d * n + 128,), 7.5, device=DEV)
    xck = xg[64:-64].view(b, nck, d, n)
    out = torch.empty_like(t["u"])
    y = torch.empty_like(t["u"]) if hz else None
    last = torch.full((b, d, n), float("nan"), device=DEV)
    ss.forward_into(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], True, out, xck, z=t["z"],
                    y=y, last_state=last, workspace=ws)
    assert ss.forward_kernel_name(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], True, out, xck,
                                  z=t["z"], y=y) == "ss_fwd_kernel_part"
    du, dd = torch.empty_like(out), torch.empty_like(out)
    dz = torch.empty_like(out) if hz else None
    g = {k: torch.full((t[r].numel() + 128,), 7.5, device=DEV) for k, r in
         (("dA", "A"), ("dB", "B"), ("dC", "C"), ("dD", "D"), ("ddelta_bias", "delta_bias"))}
    v = {k: g[k][64:-64].view(t[r].shape) for k, r in
         (("dA", "A"), ("dB", "B"), ("dC", "C"), ("dD", "D"), ("ddelta_bias", "delta_bias"))}
    args = (t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], t["dout"], xck, True, du, dd,
            v["dA"], v["dB"], v["dC"], v["dD"], v["ddelta_bias"])
    # (fp32 rows off 64-byte boundaries: the partial form of the shifted stores)
    name = "ss_bwd_fast_shift" if dt == F32 and vB and vC and n <= 16 and l % 16 else "ss_bwd_kernel_part"
    assert ss.backward_kernel_name(*args, z=t["z"], y=y, dz=dz) == name
    ss.backward_into(*args, z=t["z"], y=y, dz=dz, workspace=ws, zero_grads=True)
    torch.cuda.synchronize()
    for k, buf in dict(g, x=xg).items():
        assert (buf[:64] == 7.5).all() and (buf[-64:] == 7.5).all(), f"{k}: written outside"
    args = dict(D=x["D"], z=x["z"], delta_bias=x["delta_bias"], delta_softplus=True)
    rout, rlast = c_oracle.fwd(x["u"], x["delta"], x["A"], x["B"], x["C"], **args)
    rg = c_oracle.bwd(x["u"], x["delta"], x["A"], x["B"], x["C"], dout=x["dout"], **args)
    tol = TOL[dt]
    assert_close(out.cpu(), rout, tol, tol, "out")
    assert_close(last.cpu(), rlast, 1e-3, 1e-3, "last_state")
    assert_close(xck[:, -1].cpu(), rlast, 1e-3, 1e-3, "x")
    got = dict(v, du=du, ddelta=dd, **({"dz": dz} if hz else {}))
    for k, w in got.items():
        scale = float(torch.as_tensor(rg[k]).abs().max())
        assert_close(w.cpu(), rg[k], tol, tol * max(1.0, scale), k)
