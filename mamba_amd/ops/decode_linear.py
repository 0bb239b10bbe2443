"""Decode-size linear layer on the HIP library's matrix-core kernel.

``decode_linear(x, weight, bias=None, conv=None)`` computes
``F.linear(x, weight, bias)`` for the few rows of a single-token step (x:
(batch, k_in), weight: (n_out, k_in), nn.Linear's layout).  bf16 / fp16 rows
with k_in a multiple of 16 and unit column strides take ``ss_decode_linear``
(one pass over the weight on the matrix cores, K split over several
workgroups per output tile when there are few tiles); other shapes and
dtypes take torch's library GEMM, which computes the same product.

``conv=(conv_state, conv_weight, conv_bias, activation)`` fuses the block's
conv step into the product: outputs ``n < conv_state.shape[1]`` are replaced
by ``causal_conv1d_update`` of the product rounded to x's dtype (the conv
state advances in place), the rest are returned as they are.  This is the
block's input projection and conv update in one launch.

``norm=(residual, norm_weight, eps)`` fuses the RMSNorm in front of the
product: x is then the RMSNorm input, the product's input rows are
``rms_norm_fn(x, norm_weight, residual, eps, prenorm=True)``'s output, bit for
bit, computed in the same launch, and the call returns ``(y, s)`` with s =
x + residual (x itself without residual), the residual stream that the
prenorm RMSNorm returns.  Shapes the fused launch does not take (rows that
are not 16-byte aligned, k_in above 1024) run the RMSNorm kernel first.

The split needs a small workspace (its tile counters and fp32 partial tiles,
at most about 0.25 MiB); one is kept per (device, stream), allocated zeroed
the first time that stream calls outside a graph capture, and reused by every
later call on it, captured ones included (the kernel leaves it ready for the
next call).  A call captured on a stream that has none yet runs without the
split.  Calls that share a stream run in order, so they never use the
workspace at the same time.  Work that may run beside that stream's own
(a captured graph replayed on another stream) brings its own workspace:
``private_workspace(ws)`` makes the calls of the current thread inside it
use ``ws`` (from ``new_workspace``) instead, which is how ``GraphedStep``
gives every captured step a workspace of its own.
"""
import contextlib
import threading

import torch
import torch.nn.functional as F

from .. import _native as nat
from ..selective_scan import _raw_stream
from .causal_conv1d import _silu_flag, causal_conv1d_update

_MAX_ROWS = 64
_WS_BYTES = 1 << 20            # covers every split the library picks (at most 63 tiles x 4 slices x 1 KiB + counters)
_workspaces = {}
_ws_lock = threading.Lock()
_private = threading.local()


def new_workspace(device):
    """A zeroed split workspace, for ``private_workspace``."""
    return torch.zeros(_WS_BYTES, dtype=torch.uint8, device=device)


@contextlib.contextmanager
def private_workspace(ws):
    """Calls of this thread inside the block use ``ws`` (on its device) as
    their split workspace instead of the per-stream one."""
    prev = getattr(_private, "ws", None)
    _private.ws = ws
    try:
        yield ws
    finally:
        _private.ws = prev


def _fits(x, weight, bias):
    return nat.host().linear_fits(x, weight, bias, _MAX_ROWS)


def _workspace(device):
    """The split workspace of (device, current stream), or None while a graph
    is being captured on a stream that has none yet; inside
    ``private_workspace`` the one given there."""
    ws = getattr(_private, "ws", None)
    if ws is not None and ws.device == device:
        return ws
    stream = torch.cuda.current_stream(device)
    key = (device.index, stream.cuda_stream)
    ws = _workspaces.get(key)
    if ws is not None or torch.cuda.is_current_stream_capturing():
        return ws
    with _ws_lock:
        ws = _workspaces.get(key)
        if ws is None:
            ws = torch.zeros(_WS_BYTES, dtype=torch.uint8, device=device)
            _workspaces[key] = ws
    return ws


def decode_linear(x, weight, bias=None, conv=None, split=True, norm=None):
    """See the module docstring; ``split=False`` runs without the K split (one
    workgroup per output tile)."""
    if norm is not None:
        residual, norm_weight, eps = norm
        if not (_fits(x, weight, bias) and nat.host().linear_norm_fits(x, residual, norm_weight)):
            from .rms_norm import rms_norm_fn
            normed, s = rms_norm_fn(x, norm_weight, residual, eps, prenorm=True)
            return decode_linear(normed, weight, bias, conv=conv, split=split), s
    elif not _fits(x, weight, bias):
        y = F.linear(x, weight, bias)
        if conv is not None:
            dim = conv[0].shape[1]
            y[:, :dim] = causal_conv1d_update(y[:, :dim], *conv)
        return y
    else:
        residual = norm_weight = None
        eps = 0.0
    conv_state = conv_w = conv_b = None
    silu = False
    if conv is not None:
        conv_state, conv_w, conv_b, activation = conv
        silu = _silu_flag(activation)
    host = nat.host()
    stream = _raw_stream(x.device)
    ws = None
    if split:
        ws = getattr(_private, "ws", None)
        if ws is None or ws.device != x.device:
            ws = _workspaces.get((x.device.index, stream))
        if ws is None and host.linear_ws_bytes(x.shape[0], weight.shape[0], x.shape[1]) > 0:
            ws = _workspace(x.device)
    y, s = host.linear(x, weight, bias, conv is not None, conv_state, conv_w, conv_b, silu, norm is not None,
                       residual, norm_weight, float(eps), ws, stream)
    return (y, s) if norm is not None else y
