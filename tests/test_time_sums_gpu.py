"""The scan backward's sums over time (dA, and constant dB / dC) round often enough,
against the float64 C oracle.

The last step's terms are 2^25 times the others' (its dout is), so one running fp32 sum
over the row would drop every later one: 2000 / 2^25 = 6e-5 of the result.

* Partial blocks add a 16-step chunk's sum at a time: the 125 sums are each added with half
  a spacing of error, at most 2^-24 of the result: 7.5e-6 in all, beside about 1e-6 of the
  terms' own rounding.
* Whole blocks restart the sum after each quarter of the chunks, 30 of them here: at most
  the 480 terms of one quarter are dropped, 1.43e-5, beside four adds of 2^-24 and the
  terms' rounding.
"""
import sys

import pytest
import torch

from mamba_amd import selective_scan as ss
from oracle import c_oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("d,n,const,bound", [(24, 8, False, 1e-5), (20, 16, False, 1e-5), (24, 8, True, 1e-5),
                                             (24, 5, True, 1e-5), (32, 16, False, 1.7e-5), (16, 16, True, 1.7e-5)])
def test_sums_over_time(d, n, const, bound):
    l = 2000
    print(f"\n[time sums] dim {d} dstate {n} constant {const}", flush=True)
    sys.stdout.flush()
    one = torch.ones(1, d, l)
    u, dout = one.clone(), one.clone()
    dout[..., -1] = 2.0 ** 25
    delta = one * 0.25
    A = -8.0 - torch.arange(d * n).view(d, n) / float(d * n)         # a = exp(0.25 A): about 1 / 8
    B = C = torch.ones(d, n) if const else torch.ones(1, 1, n, l)
    t = [v.to(DEV) for v in (u, delta, A, B, C)]
    out, xck = torch.empty_like(t[0]), torch.empty((1, ss.n_chunks(l), d, n), device=DEV)
    ss.forward_into(*t, None, None, False, out, xck, workspace=None)
    g = [torch.empty_like(v) for v in t]
    ss.backward_into(*t, None, None, dout.to(DEV), xck, False, *g, None, None, workspace=None, zero_grads=True)
    ref = c_oracle.bwd(u, delta, A, B, C, dout=dout, delta_softplus=False)
    for k, w in (("dA", g[2]),) + ((("dB", g[3]), ("dC", g[4])) if const else ()):
        r = torch.as_tensor(ref[k]).double()
        err = float((w.cpu().double() - r).norm() / r.norm())
        assert err < bound, (k, err)
