"""The decode-size linear layer at the edges of its launch shapes: K steps
around the 4-, 8- and 16-wave launches and one to five steps per wave, 16- and
32-wide steps, a K slice shorter than the others, tails in n and batch, with
and without the fused RMSNorm.  Against the product in float64 of the same
rounded inputs: fp32 sums of at most 5120 terms of size k^-1/2 are within
1e-4 of it, and the result is rounded once to bf16 (at most 2^-8 of its size).
"""
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
K = [16, 32, 48, 64, 128, 160, 256, 272, 288, 512, 528, 544, 1024, 1056, 2048, 2080, 5120]


@pytest.mark.parametrize("k", K)
@pytest.mark.parametrize("split", [False, True], ids=["whole", "split"])
def test_wave_and_step_edges(k, split):
    from mamba_amd.ops import decode_linear as dlm
    from mamba_amd.ops.rms_norm import rms_norm_fn
    print(f"\n[decode linear] k {k} split {split}", flush=True)
    sys.stdout.flush()
    gen = torch.Generator().manual_seed(k)
    for batch, n in ((1, 16), (17, 33)):
        x = torch.randn(batch, k, generator=gen).bfloat16().to(DEV)
        w = (torch.randn(n, k, generator=gen) / k ** 0.5).bfloat16().to(DEV)
        y = dlm.decode_linear(x, w, split=split).double()
        ref = x.double() @ w.double().t()
        assert (y - ref).abs().le(2.0 ** -8 * ref.abs() + 1e-4).all()
        if k <= 1024 and not split:
            r = torch.randn(batch, k, generator=gen).bfloat16().to(DEV)
            nw = (torch.randn(k, generator=gen) * 0.1).bfloat16().to(DEV)
            yf, s = dlm.decode_linear(x, w, norm=(r, nw, 1e-6))
            normed, s0 = rms_norm_fn(x, nw, r, prenorm=True)
            assert torch.equal(s, s0)
            assert torch.equal(yf, dlm.decode_linear(normed, w, split=False))


def test_missing_tensors_are_refused():
    """None where a tensor is needed raises (before any launch), in the fused conv step of
    the linear layer and in the state update."""
    from mamba_amd.ops import decode_linear as dlm
    from mamba_amd.ops.selective_state_update import selective_state_update
    print("\n[decode] missing tensors", flush=True)
    sys.stdout.flush()
    x, w = torch.zeros(2, 32, device=DEV).bfloat16(), torch.zeros(48, 32, device=DEV).bfloat16()
    state, taps = torch.zeros(2, 16, 4, device=DEV).bfloat16(), torch.zeros(16, 4, device=DEV)
    for conv in ((None, taps, None, "silu"), (state, None, None, None)):
        with pytest.raises(ValueError, match="required"):
            dlm.decode_linear(x, w, conv=conv)
    ssm, u, A, B = torch.zeros(2, 32, 16, device=DEV), x, torch.zeros(32, 16, device=DEV), x[:, :16]
    for dt in (None, (x[:, :4], None)):
        with pytest.raises(ValueError, match="required"):
            selective_state_update(ssm, u, dt, A, B, B)
