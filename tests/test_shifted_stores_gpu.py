"""fp32 backward into rows off 64-byte boundaries: each 16-step chunk's du,
ddelta and dz are stored one 64-byte block of the row at a time, part of it a
chunk late.  Against the same call into rows on those boundaries, which stores
whole chunks: the same bits (both kernels compute the same values; only the
stores differ), and nothing outside the rows is written.

Offsets put the boundary at every kind of place, differently for the three
arrays; seqlens sit around one and two chunks and chunk pairs, and long enough
for sequence segments; 40 channels end in a partial block.
"""
import sys

import pytest
import torch

from mamba_amd import selective_scan as ss
from oracle.selective_scan_ref import make_inputs

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _view(batch, dim, seqlen, offset, row):
    """(batch, dim, seqlen) view `offset` floats into a buffer of NaNs, rows `row` floats apart."""
    buf = torch.full((offset + batch * dim * row + 64,), float("nan"), device=DEV)
    return buf, buf[offset:offset + batch * dim * row].view(batch, dim, row)[..., :seqlen]


@pytest.mark.parametrize("seqlen", [1, 15, 16, 17, 31, 32, 33, 48, 63, 65, 100, 1030])
@pytest.mark.parametrize("dim,has_z", [(32, True), (40, False)])
def test_shifted_rows_give_the_same_bits(seqlen, dim, has_z):
    print(f"\n[shift] seqlen {seqlen} dim {dim} z {has_z}", flush=True)
    sys.stdout.flush()
    batch, n = 2, 16
    x = make_inputs(batch, dim, n, seqlen, seed=50 + seqlen, has_z=has_z)
    t = {k: v.to(DEV) if v is not None else None for k, v in x.items()}
    out, xck = torch.empty_like(t["u"]), torch.empty((batch, ss.n_chunks(seqlen), dim, n), device=DEV)
    y = torch.empty_like(out) if has_z else None
    ss.forward_into(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], True, out, xck, z=t["z"], y=y)

    def run(layout):
        bufs = [_view(batch, dim, seqlen, *p) for p in layout]
        g = {k: torch.empty(t[r].shape, device=DEV) for k, r in
             (("dA", "A"), ("dB", "B"), ("dC", "C"), ("dD", "D"), ("db", "delta_bias"))}
        args = (t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], t["dout"], xck, True,
                bufs[0][1], bufs[1][1], g["dA"], g["dB"], g["dC"], g["dD"], g["db"])
        grads = dict(z=t["z"], y=y, dz=bufs[2][1] if has_z else None)
        off64 = any(offset % 16 or row % 16 for offset, row in layout[:3 if has_z else 2])
        assert ss.backward_kernel_name(*args, **grads) == ("ss_bwd_fast_shift" if off64 else "ss_bwd_fast"
                                                           if dim % 16 == 0 else "ss_bwd_kernel_part")
        ss.backward_into(*args, **grads, zero_grads=True)
        torch.cuda.synchronize()
        used = bufs if has_z else bufs[:2]
        for buf, v in used:
            assert torch.isfinite(v).all()
            assert int(torch.isnan(buf).sum()) == buf.numel() - v.numel(), "written outside the rows"
        return [v.clone() for _, v in used]

    pad = (seqlen + 15) // 16 * 16
    want = run([(0, pad)] * 3)                                     # rows on 64-byte boundaries
    for layout in ([(1, pad), (15, pad), (8, pad)], [(0, pad + 1), (3, pad + 7), (0, pad)],
                   [(0, seqlen), (0, seqlen), (5, pad + 3)]):
        for a, b in zip(want, run(layout)):
            assert torch.equal(a, b)
