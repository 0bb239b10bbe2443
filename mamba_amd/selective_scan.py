"""Drop-in for the reference's native module ``selective_scan``.

The reference builds a pybind extension named ``selective_scan``
(setup.py:10-16, csrc/selective_scan/selective_scan.cpp:331-334) with

    forward(u, delta, A, B, C, D, delta_bias, use_delta_softplus) -> [out, x]
    backward(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus)
        -> [du, ddelta, dA, dB, dC, dD, ddelta_bias]

This module keeps those positional signatures and return lists and runs
them on libmamba_ss.so through its C ABI.  Host-side rules mirror
selective_scan.cpp:184-329: B (or C) with fewer than 3 dims is constant
(dim, dstate) (:194-195); n_groups = B.size(1) (:202); out has delta's
dtype (:206); du / ddelta have the dtypes of u / delta, dA / dD /
ddelta_bias are zero-initialised fp32 accumulators and variable dB / dC are
fp32 (:271-287).  Unlike the reference, inputs are validated, and a fused z
gate is available through the keyword-only ``z`` (forward then also returns
the pre-gate output y, which ``backward`` needs to produce dz).

There is no CPU fallback: tensors must live on a ROCm device and the
library must be built.
"""
import ctypes

import torch

from . import _native as nat

_ITYPES = {torch.float32: nat.SS_F32, torch.bfloat16: nat.SS_BF16, torch.float16: nat.SS_F16}


def chunk_size():
    """Steps per checkpoint of the state h in x."""
    return int(nat.load().ss_chunk_size())


def n_chunks(seqlen):
    cs = chunk_size()
    return (seqlen + cs - 1) // cs


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _require(cond, msg):
    if not cond:
        raise ValueError(f"selective_scan: {msg}")


def _raw_stream(device):
    """The device's current stream as an integer handle (0 for a device that is no GPU,
    which the calls it is passed to refuse)."""
    return torch._C._cuda_getCurrentRawStream(device.index) if device.type == "cuda" else 0


def _stream(device):
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def _fwd_into_args(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, z, y, last_state=None):
    a = nat.FwdArgs()
    nat.host().fill_fwd_into(ctypes.addressof(a), u, delta, A, B, C, D, delta_bias, bool(use_delta_softplus), out, x,
                             z, y, last_state)
    return a


def _attach_fwd_workspace(lib, a, workspace, device):
    """Sets the forward's optional workspace: "auto" allocates what the library
    asks for (torch's caching allocator; none for most shapes), a tensor is
    used as given, None runs the serial scan.  Returns the tensor to keep."""
    if isinstance(workspace, str):
        _require(workspace == "auto", f"workspace must be 'auto', None or a tensor, got {workspace!r}")
        n = int(lib.ss_fwd_workspace_bytes(ctypes.byref(a)))
        if n < 0:
            nat.check(nat.SS_ERR_INVALID, "selective_scan.forward")
        workspace = torch.empty(n, dtype=torch.uint8, device=device) if n > 0 else None
    if workspace is not None:
        _require(workspace.is_cuda and workspace.is_contiguous(), "workspace must be a contiguous GPU tensor")
        a.workspace, a.workspace_bytes = _ptr(workspace), workspace.numel() * workspace.element_size()
    return workspace


def forward_into(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, *, z=None, y=None,
                 last_state=None, workspace="auto"):
    """Forward into caller-allocated ``out`` (delta's dtype), ``x`` (fp32
    (batch, n_chunks, dim, dstate) contiguous) and, with ``z``, ``y``.

    ``x`` and ``y`` are what the backward needs; either may be None for a
    forward that no backward follows (they are then not written at all).
    ``last_state`` (fp32 (batch, dim, dstate), optional) receives the state
    after the last step.  ``workspace`` ("auto", a tensor or None) lets a
    forward with few (batch, channel) rows scan sequence segments in
    parallel (see ``forward_workspace_bytes``)."""
    auto = isinstance(workspace, str)
    if auto:
        _require(workspace == "auto", f"workspace must be 'auto', None or a tensor, got {workspace!r}")
    nat.host().scan_fwd(u, delta, A, B, C, D, delta_bias, bool(use_delta_softplus), out, x, z, y, last_state,
                        auto, None if auto else workspace, _raw_stream(u.device))


def forward_workspace_bytes(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, *, z=None, y=None):
    """Bytes of scratch ``forward_into`` can use for these tensors (0: none;
    nonzero when the batch has too few channel rows to fill the GPU and the
    sequence is long enough to cut into segments)."""
    lib = nat.load()
    a = _fwd_into_args(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, z, y)
    n = lib.ss_fwd_workspace_bytes(ctypes.byref(a))
    if n < 0:
        nat.check(nat.SS_ERR_INVALID, "selective_scan.forward_workspace_bytes")
    return int(n)


def prepare_forward(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, *, z=None, y=None,
                    last_state=None, workspace="auto"):
    """Validates the arguments of ``forward_into`` once and returns a callable
    that launches the same forward again, on the stream that is current now,
    with no host-side work beyond the C call (the tensors must stay alive
    and keep their storage).  For repeated launches over fixed buffers."""
    lib = nat.load()
    a = _fwd_into_args(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, z, y, last_state)
    ws = _attach_fwd_workspace(lib, a, workspace, u.device)
    dev = u.device
    stream = torch.cuda.current_stream(dev)
    handle = ctypes.c_void_p(stream.cuda_stream)
    ref = ctypes.byref(a)

    def launch():
        nat.check(lib.ss_fwd(ref, handle), "selective_scan.forward")
    launch.args = a
    launch.workspace = ws
    return launch


def forward_kernel_name(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, *, z=None, y=None):
    """Base name of the kernel ``forward_into`` launches for these tensors
    ("" when there is no work).  No device work."""
    lib = nat.load()
    a = _fwd_into_args(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, z, y)
    name = lib.ss_fwd_kernel_name(ctypes.byref(a))
    if name is None:
        nat.check(nat.SS_ERR_INVALID, "selective_scan.forward_kernel_name")
    return name.decode()


def forward(u, delta, A, B, C, D=None, delta_bias=None, use_delta_softplus=True, *, z=None):
    """selective_scan.forward (selective_scan.cpp:184-244).

    Returns [out, x]; with ``z`` given, [out, x, y] where out = y * silu(z)
    and y is the pre-gate output saved for ``backward``.
    """
    batch, dim, seqlen = u.shape
    dstate = A.shape[1]
    out = torch.empty_like(delta, memory_format=torch.contiguous_format)
    x = torch.empty((batch, n_chunks(seqlen), dim, dstate), dtype=torch.float32, device=u.device)
    y = torch.empty_like(out) if z is not None else None
    forward_into(u, delta, A, B, C, D, delta_bias, use_delta_softplus, out, x, z=z, y=y)
    return [out, x] if z is None else [out, x, y]


def _bwd_into_args(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                   du, ddelta, dA, dB, dC, dD, ddelta_bias, z, y, dz):
    b = nat.BwdArgs()
    nat.host().fill_bwd(ctypes.addressof(b), u, delta, A, B, C, D, delta_bias, dout, x, bool(use_delta_softplus),
                        du, ddelta, dA, dB, dC, dD, ddelta_bias, z, y, dz)
    return b


def workspace_bytes(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                    du, ddelta, dA, dB, dC, dD, ddelta_bias, *, z=None, y=None, dz=None, deterministic=None):
    """Bytes of scratch ``backward_into`` can use for these tensors (0: none)."""
    lib = nat.load()
    b = _bwd_into_args(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                       du, ddelta, dA, dB, dC, dD, ddelta_bias, z, y, dz)
    _set_deterministic(lib, b, deterministic)
    n = lib.ss_bwd_workspace_bytes(ctypes.byref(b))
    if n < 0:
        nat.check(nat.SS_ERR_INVALID, "selective_scan.workspace_bytes")
    return int(n)


def _set_deterministic(lib, b, flag, workspace="auto"):
    """Sets b.deterministic: the flag, or with None torch.use_deterministic_algorithms.
    An explicit request the kernels cannot honour raises (from the library);
    one that comes from torch's setting raises as torch's own ops do, or
    warns and runs with atomic sums under warn_only.  The deterministic sums
    need a workspace: a call made with ``workspace=None`` cannot have them."""
    if flag is not None:
        b.deterministic = int(bool(flag))
        return
    b.deterministic = int(torch.are_deterministic_algorithms_enabled())
    if not b.deterministic:
        return
    msg = None
    if lib.ss_bwd_workspace_bytes(ctypes.byref(b)) < 0:
        msg = ("selective_scan.backward has no deterministic implementation for these arguments: "
               + lib.ss_last_error().decode())
    elif workspace is None:
        msg = ("selective_scan.backward: the deterministic sums need a workspace, and this call passes "
               "workspace=None")
    if msg is not None:
        if not torch.is_deterministic_algorithms_warn_only_enabled():
            raise RuntimeError(msg)
        import warnings
        warnings.warn(msg)
        b.deterministic = 0


def backward_into(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                  du, ddelta, dA, dB, dC, dD, ddelta_bias, *, z=None, y=None, dz=None, workspace="auto",
                  zero_grads=False, deterministic=None):
    """Backward into caller-allocated gradients.  du, ddelta (and dz) are
    overwritten; dA, dB, dC, dD, ddelta_bias are fp32 and accumulated into,
    or, with ``zero_grads``, cleared by the library first (their contents on
    entry are ignored, so ``torch.empty`` buffers will do).

    ``workspace``: "auto" allocates the scratch the library asks for (see
    ``workspace_bytes``) from torch's caching allocator; a uint8 / any CUDA
    tensor is used as given; None runs without one (same results).

    ``deterministic``: sum dB, dC, dA, dD and ddelta_bias in a fixed order
    (the same bits on every run; needs the fast kernels and a workspace);
    None follows ``torch.use_deterministic_algorithms``.
    """
    auto = isinstance(workspace, str)
    if auto:
        _require(workspace == "auto", f"workspace must be 'auto', None or a tensor, got {workspace!r}")
    if deterministic is None and torch.are_deterministic_algorithms_enabled():
        b = _bwd_into_args(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                           du, ddelta, dA, dB, dC, dD, ddelta_bias, z, y, dz)
        _set_deterministic(nat.load(), b, None, workspace)
        deterministic = bool(b.deterministic)
    nat.host().scan_bwd(u, delta, A, B, C, D, delta_bias, dout, x, bool(use_delta_softplus),
                        du, ddelta, dA, dB, dC, dD, ddelta_bias, z, y, dz,
                        auto, None if auto else workspace, bool(zero_grads), bool(deterministic),
                        _raw_stream(u.device))


def prepare_backward(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                     du, ddelta, dA, dB, dC, dD, ddelta_bias, *, z=None, y=None, dz=None, workspace="auto",
                     zero_grads=False, deterministic=None):
    """``backward_into`` validated once, as a callable that relaunches it on
    the stream that is current now (see ``prepare_forward``); the workspace,
    if any, is allocated here and kept by the callable."""
    lib = nat.load()
    b = _bwd_into_args(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                       du, ddelta, dA, dB, dC, dD, ddelta_bias, z, y, dz)
    _set_deterministic(lib, b, deterministic, workspace)
    if isinstance(workspace, str):
        _require(workspace == "auto", f"workspace must be 'auto', None or a tensor, got {workspace!r}")
        n = lib.ss_bwd_workspace_bytes(ctypes.byref(b))
        if n < 0:
            nat.check(nat.SS_ERR_INVALID, "selective_scan.backward")
        workspace = torch.empty(n, dtype=torch.uint8, device=u.device) if n > 0 else None
    if workspace is not None:
        _require(workspace.device == u.device and workspace.is_contiguous(),
                 "workspace must be a contiguous tensor on the inputs' device")
        b.workspace = _ptr(workspace)
        b.workspace_bytes = workspace.numel() * workspace.element_size()
    b.zero_grads = int(bool(zero_grads))
    stream = torch.cuda.current_stream(u.device)
    handle = ctypes.c_void_p(stream.cuda_stream)
    ref = ctypes.byref(b)

    def launch():
        nat.check(lib.ss_bwd(ref, handle), "selective_scan.backward")
    launch.args = b
    launch.workspace = workspace
    return launch


def backward_kernel_name(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                         du, ddelta, dA, dB, dC, dD, ddelta_bias, *, z=None, y=None, dz=None):
    """Base name of the kernel ``backward_into`` launches for these tensors
    ("" when there is no work).  No device work."""
    lib = nat.load()
    b = _bwd_into_args(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                       du, ddelta, dA, dB, dC, dD, ddelta_bias, z, y, dz)
    name = lib.ss_bwd_kernel_name(ctypes.byref(b))
    if name is None:
        nat.check(nat.SS_ERR_INVALID, "selective_scan.backward_kernel_name")
    return name.decode()


def backward(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus, *, z=None, y=None):
    """selective_scan.backward (selective_scan.cpp:246-329).

    Returns [du, ddelta, dA, dB, dC, dD, ddelta_bias]; with ``z`` (and the
    forward's ``y``) also dz as an eighth entry.
    """
    if not torch.are_deterministic_algorithms_enabled():
        res = nat.host().scan_bwd_new(u, delta, A, B, C, D, delta_bias, dout, x, bool(use_delta_softplus), z, y,
                                      False, _raw_stream(u.device))
        return list(res if z is not None else res[:7])
    du = torch.empty_like(u, memory_format=torch.contiguous_format)
    ddelta = torch.empty_like(delta, memory_format=torch.contiguous_format)
    # the accumulators are cleared by the library in the launch that clears
    # its workspace (zero_grads), not by separate torch fills
    dA = torch.empty(A.shape, dtype=torch.float32, device=A.device)
    dB = torch.empty(B.shape, dtype=torch.float32, device=B.device)
    dC = torch.empty(C.shape, dtype=torch.float32, device=C.device)
    dD = torch.empty(D.shape, dtype=torch.float32, device=D.device) if D is not None else None
    ddelta_bias = (torch.empty(delta_bias.shape, dtype=torch.float32, device=delta_bias.device)
                   if delta_bias is not None else None)
    dz = torch.empty_like(z, memory_format=torch.contiguous_format) if z is not None else None
    backward_into(u, delta, A, B, C, D, delta_bias, dout, x, use_delta_softplus,
                  du, ddelta, dA, dB, dC, dD, ddelta_bias, z=z, y=y, dz=dz, zero_grads=True)
    res = [du, ddelta, dA, dB, dC, dD, ddelta_bias]
    if z is not None:
        res.append(dz)
    return res
