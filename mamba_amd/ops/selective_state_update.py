"""One decode step of the selective scan on the HIP library.

``selective_state_update(state, x, dt, A, B, C, D=None, z=None, dt_bias=None,
dt_softplus=False)`` advances the scan of forward_kernel.cu:216-293 by one
token from a state kept between tokens (the reference has no decode path:
CausalLM.generate is a stub, models/causal_lm.py:61-62):

    dt' = softplus(dt + dt_bias)
    state[b, d, n] <- exp(dt' A[d, n]) state[b, d, n] + dt' x[b, d] B[b, g, n]   (in place, fp32)
    out[b, d] = sum_n C[b, g, n] state[b, d, n] + D[d] x[b, d], times silu(z[b, d])

state: fp32 (batch, dim, dstate); x, dt, z: (batch, dim); A: (dim, dstate);
B, C: (batch, dstate) or (batch, n_groups, dstate), in x's dtype (any
strides); D, dt_bias: (dim,).  Returns out (batch, dim) in x's dtype.

dt may also be a pair (dt_low, dt_weight): the block's delta projection
dt = dt_low @ dt_weight.T (modules/mamba_simple.py:118-119), with dt_low
(batch, rank) and dt_weight (dim, rank) in x's dtype, summed in fp32 inside
the kernel, so a decode step needs no launch for that product.
"""
from .. import _native as nat
from ..selective_scan import _raw_stream


def selective_state_update(state, x, dt, A, B, C, D=None, z=None, dt_bias=None, dt_softplus=False, out=None):
    low, w = dt if isinstance(dt, (tuple, list)) else (None, None)
    return nat.host().state_update(state, x, None if low is not None else dt, low, w, A, B, C, D, z, dt_bias,
                                   bool(dt_softplus), out, _raw_stream(x.device))
