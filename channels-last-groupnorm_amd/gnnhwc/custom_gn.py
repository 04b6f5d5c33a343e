"""Python surface of the NHWC GroupNorm op: ``GN_NHWC`` (an ``nn.GroupNorm`` subclass with a fused
activation), its ``autograd.Function`` and the ``gnop::fwd`` / ``gnop::bwd`` operators.

Mirrors src/gnnhwc/custom_gn.py:29-90 and the operator glue src/gnnhwc/csrc/custom_gn.cpp:10-94 of the
reference; the kernels behind the operators are the HIP ones in libgnnhwc_hip.so, reached through its
C ABI (include/gnnhwc.h) with raw device pointers and the current HIP stream.  torch only provides
device memory (outputs, workspace) and the stream.
"""
import collections
import threading

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _cabi, _native

_DTYPE_CODE = {
    torch.float32: _cabi.F32,
    torch.float64: _cabi.F64,
    torch.float16: _cabi.F16,
    torch.bfloat16: _cabi.BF16,
}

# custom_gn.py:52-59
ACTIVATION_CODES = {
    "identity": 0,
    "relu": 1,
    "swish": 2,
    "silu": 2,
    "gelu": 3,
    "gelu_tanh": 4,
}


def _check_device(t, name):
    # CHECK_CUDA, custom_gn.cpp:8,17-19,53-58 (a ROCm build of torch calls the HIP device "cuda")
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)


def _dtype_code(t, name):
    try:
        return _DTYPE_CODE[t.dtype]
    except KeyError:
        # AT_DISPATCH_FLOATING_TYPES_AND2 raises for any other type (custom_gn.cpp:29-33)
        raise RuntimeError('"group_norm_nhwc" not implemented for %s (%s)' % (t.dtype, name)) from None


def _stats_dtype(x_dtype):
    # The reference allocates mean / rstd in the parameters' (= data's) dtype (custom_gn.cpp:26-27).
    # For 16-bit data that rounding would leak into dx, so statistics are kept in float32 there.
    return torch.float32 if x_dtype in (torch.float16, torch.bfloat16) else x_dtype


def _as_nrc(t):
    """(N, C, R) tensor with strides (R*C, 1, C) -> contiguous (N, R, C) view (copies only if it must)."""
    t = t.permute(0, 2, 1)
    return t if t.is_contiguous() else t.contiguous()


def _param_args(weight, bias, C, data_code):
    """(param dtype code, weight pointer, bias pointer, tensors to keep alive) for the C ABI.  weight and bias are
    either both tensors of C elements on the device and of one dtype, or both None: the C ABI takes NULL for
    gamma = 1, beta = 0, so a normalisation without parameters never materialises ones and zeros
    (the reference does, custom_gn.py:83-86)."""
    if weight is None and bias is None:
        return data_code, None, None, ()
    if weight is None or bias is None:
        raise RuntimeError("weight and bias must both be given or both be None")
    _check_device(weight, "weight")
    _check_device(bias, "bias")
    if bias.dtype != weight.dtype:
        raise RuntimeError("weight and bias must have the same dtype (%s vs %s)" % (weight.dtype, bias.dtype))
    if weight.numel() != C or bias.numel() != C:
        raise RuntimeError("weight and bias must have %d elements" % C)
    w, b = weight.contiguous(), bias.contiguous()
    return _dtype_code(weight, "weight"), w.data_ptr(), b.data_ptr(), (w, b)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _current_stream_ptr(device):
    """hipStream_t of torch's current stream on `device` (the raw getter is an order of magnitude cheaper than
    building a torch.cuda.Stream object on every call)."""
    if _raw_stream is not None:
        return _raw_stream(device.index)
    return torch.cuda.current_stream(device).cuda_stream


class _on_device:
    """Makes `device` current for the C ABI call (the reference has no device guard, custom_gn.cpp:10-42); does
    nothing when it already is, which is the usual case and keeps the context manager off the hot path."""

    __slots__ = ("guard",)

    def __init__(self, device):
        self.guard = None if device.index == torch.cuda.current_device() else torch.cuda.device(device)

    def __enter__(self):
        if self.guard is not None:
            self.guard.__enter__()

    def __exit__(self, *exc):
        if self.guard is not None:
            self.guard.__exit__(*exc)
        return False


_workspaces = collections.OrderedDict()
_workspaces_lock = threading.Lock()
_MAX_CACHED_WORKSPACES = 8


def _workspace(nbytes, device, stream_ptr):
    """Scratch memory for one call.  Calls on one stream follow each other, so they can share one buffer per
    (device, stream), grown on demand; while the stream is recording a graph the buffer comes from the allocator
    instead (it then belongs to the graph's own memory pool, like every other tensor of the capture).
    The cache is shared by the caller's thread and the autograd engine's, hence the lock; it keeps the buffers of the
    most recently used streams only, so that streams that no longer exist do not pin memory for ever (a buffer that is
    dropped while a kernel still uses it stays valid: the caching allocator only reuses it in stream order)."""
    if torch.cuda.is_current_stream_capturing():
        return torch.empty((nbytes,), dtype=torch.uint8, device=device)
    key = (device.index, stream_ptr)
    with _workspaces_lock:
        ws = _workspaces.get(key)
        if ws is None or ws.numel() < nbytes:
            ws = torch.empty((max(nbytes, 1 << 20),), dtype=torch.uint8, device=device)
            _workspaces[key] = ws
        _workspaces.move_to_end(key)
        while len(_workspaces) > _MAX_CACHED_WORKSPACES:
            _workspaces.popitem(last=False)
    return ws


def gn_nhwc_fwd(X, weight, bias, G, eps, act_fn_option):
    """gnop::fwd -- custom_gn.cpp:10-42.  X: (N, C, R) channels-last view.  Returns (Y, means, rstds)."""
    return _nhwc_fwd(X, weight, bias, G, eps, act_fn_option, None, "gnop::fwd")


def gn_nhwc_fwd_cast(X, weight, bias, G, eps, act_fn_option, out_dtype):
    """gnop::fwd_cast (no counterpart in the reference, whose Y has X's dtype, custom_gn.cpp:28): gnop::fwd on float32
    data with Y written as float16 / bfloat16 by the kernel itself, for a consumer that runs in half precision."""
    return _nhwc_fwd(X, weight, bias, G, eps, act_fn_option, out_dtype, "gnop::fwd_cast")


def _nhwc_fwd(X, weight, bias, G, eps, act_fn_option, out_dtype, opname):
    _check_device(X, "X")
    if X.dim() != 3:
        raise RuntimeError("%s expects X of shape (N, C, R), got %s" % (opname, tuple(X.shape)))
    N, C, R = X.shape
    dt = _dtype_code(X, "X")
    pdt, w_ptr, b_ptr, _keep = _param_args(weight, bias, C, dt)
    X_nrc = _as_nrc(X)
    if out_dtype is None or out_dtype == X.dtype:
        Y = torch.empty_like(X_nrc)
    elif X.dtype == torch.float32 and out_dtype in (torch.float16, torch.bfloat16):
        Y = torch.empty(X_nrc.shape, dtype=out_dtype, device=X.device)
    else:
        raise RuntimeError("%s: out_dtype %s with %s data (float32 data may leave as float16 or bfloat16)"
                           % (opname, out_dtype, X.dtype))
    sdtype = _stats_dtype(X.dtype)
    means = torch.empty((N, G), dtype=sdtype, device=X.device)
    rstds = torch.empty((N, G), dtype=sdtype, device=X.device)
    lib = _cabi.lib
    with _on_device(X.device):
        nbytes = lib.gnnhwc_fwd_workspace_bytes(N, R, C, G, dt)
        if nbytes == 0:
            raise RuntimeError(opname + ": " + _cabi.last_error())
        stream = _current_stream_ptr(X.device)
        ws = _workspace(nbytes, X.device, stream)
        rc = lib.gnnhwc_fwd_cast(
            X_nrc.data_ptr(), w_ptr, b_ptr,
            Y.data_ptr(), means.data_ptr(), rstds.data_ptr(),
            N, R, C, G, float(eps), int(act_fn_option), dt, pdt, _DTYPE_CODE[sdtype], _DTYPE_CODE[Y.dtype],
            ws.data_ptr(), ws.numel(), stream)
    _cabi.check(rc, opname)
    return Y.permute(0, 2, 1), means, rstds


def gn_nhwc_bwd(dy, X, weight, bias, means, rstds, G, act_fn_option):
    """gnop::bwd -- custom_gn.cpp:44-89.  Returns (dX (N, C, R) channels-last view, dweight, dbias)."""
    for t, name in ((dy, "dy"), (X, "X"), (means, "means"), (rstds, "rstds")):
        _check_device(t, name)
    if X.dim() != 3 or dy.shape != X.shape:
        raise RuntimeError("gnop::bwd expects dy and X of the same shape (N, C, R), got %s and %s"
                           % (tuple(dy.shape), tuple(X.shape)))
    N, C, R = X.shape
    dt = _dtype_code(X, "X")
    pdt, w_ptr, b_ptr, _keep = _param_args(weight, bias, C, dt)
    sdt = _dtype_code(means, "means")
    # (float data may come with a 16-bit gradient: the backward of gnop::fwd_cast; the kernels widen it as they load it)
    dy16 = X.dtype == torch.float32 and dy.dtype in (torch.float16, torch.bfloat16)
    if dy.dtype != X.dtype and not dy16:
        raise RuntimeError("dy and X must have the same dtype, or dy float16 / bfloat16 with float32 X (%s vs %s)" % (dy.dtype, X.dtype))
    if rstds.dtype != means.dtype:
        raise RuntimeError("means and rstds must share a dtype")
    if means.numel() != N * G or rstds.numel() != N * G:
        raise RuntimeError("means and rstds must have N*G = %d elements" % (N * G))
    X_nrc = _as_nrc(X)
    dy_nrc = _as_nrc(dy)
    dX = torch.empty_like(X_nrc)
    # a normalisation without parameters has no parameter gradients: nothing is allocated or computed for them
    dweight = torch.empty((C,), dtype=weight.dtype, device=X.device) if weight is not None else None
    dbias = torch.empty((C,), dtype=bias.dtype, device=X.device) if bias is not None else None
    lib = _cabi.lib
    with _on_device(X.device):
        nbytes = lib.gnnhwc_bwd_workspace_bytes(N, R, C, G, dt)
        if nbytes == 0:
            raise RuntimeError("gnop::bwd: " + _cabi.last_error())
        stream = _current_stream_ptr(X.device)
        ws = _workspace(nbytes, X.device, stream)
        rc = lib.gnnhwc_bwd_cast(
            dy_nrc.data_ptr(), X_nrc.data_ptr(), w_ptr, b_ptr,
            means.contiguous().data_ptr(), rstds.contiguous().data_ptr(),
            dX.data_ptr(), dweight.data_ptr() if dweight is not None else None, dbias.data_ptr() if dbias is not None else None,
            N, R, C, G, int(act_fn_option), dt, pdt, sdt, _dtype_code(dy, "dy"),
            ws.data_ptr(), ws.numel(), stream)
    _cabi.check(rc, "gnop::bwd")
    return dX.permute(0, 2, 1), dweight, dbias


def gn_nchw_fwd(X, weight, bias, G, eps, act_fn_option):
    """gnop::fwd_nchw (no counterpart in the reference, which hands channels-first input to torch,
    custom_gn.py:75-79): X is (N, C, R) contiguous.  Returns (Y contiguous like X, means, rstds)."""
    _check_device(X, "X")
    if X.dim() != 3:
        raise RuntimeError("gnop::fwd_nchw expects X of shape (N, C, R), got %s" % (tuple(X.shape),))
    N, C, R = X.shape
    dt = _dtype_code(X, "X")
    pdt, w_ptr, b_ptr, _keep = _param_args(weight, bias, C, dt)
    X = X.contiguous()
    Y = torch.empty_like(X)
    sdtype = _stats_dtype(X.dtype)
    means = torch.empty((N, G), dtype=sdtype, device=X.device)
    rstds = torch.empty((N, G), dtype=sdtype, device=X.device)
    lib = _cabi.lib
    with _on_device(X.device):
        nbytes = lib.gnnhwc_nchw_workspace_bytes(N, C, R, G, dt, 0)
        if nbytes == 0:
            raise RuntimeError("gnop::fwd_nchw: " + _cabi.last_error())
        stream = _current_stream_ptr(X.device)
        ws = _workspace(nbytes, X.device, stream)
        rc = lib.gnnhwc_fwd_nchw(
            X.data_ptr(), w_ptr, b_ptr,
            Y.data_ptr(), means.data_ptr(), rstds.data_ptr(),
            N, C, R, G, float(eps), int(act_fn_option), dt, pdt, _DTYPE_CODE[sdtype],
            ws.data_ptr(), ws.numel(), stream)
    _cabi.check(rc, "gnop::fwd_nchw")
    return Y, means, rstds


def gn_nchw_bwd(dy, X, weight, bias, means, rstds, G, act_fn_option):
    """gnop::bwd_nchw: dy, X (N, C, R) contiguous.  Returns (dX, dweight, dbias)."""
    for t, name in ((dy, "dy"), (X, "X"), (means, "means"), (rstds, "rstds")):
        _check_device(t, name)
    if X.dim() != 3 or dy.shape != X.shape:
        raise RuntimeError("gnop::bwd_nchw expects dy and X of the same shape (N, C, R), got %s and %s"
                           % (tuple(dy.shape), tuple(X.shape)))
    N, C, R = X.shape
    dt = _dtype_code(X, "X")
    pdt, w_ptr, b_ptr, _keep = _param_args(weight, bias, C, dt)
    sdt = _dtype_code(means, "means")
    # (float data may come with a 16-bit gradient: the backward of gnop::fwd_cast; the kernels widen it as they load it)
    dy16 = X.dtype == torch.float32 and dy.dtype in (torch.float16, torch.bfloat16)
    if dy.dtype != X.dtype and not dy16:
        raise RuntimeError("dy and X must have the same dtype, or dy float16 / bfloat16 with float32 X (%s vs %s)" % (dy.dtype, X.dtype))
    if rstds.dtype != means.dtype:
        raise RuntimeError("means and rstds must share a dtype")
    if means.numel() != N * G or rstds.numel() != N * G:
        raise RuntimeError("means and rstds must have N*G = %d elements" % (N * G))
    X = X.contiguous()
    dy = dy.contiguous()
    dX = torch.empty_like(X)
    dweight = torch.empty((C,), dtype=weight.dtype, device=X.device) if weight is not None else None
    dbias = torch.empty((C,), dtype=bias.dtype, device=X.device) if bias is not None else None
    lib = _cabi.lib
    with _on_device(X.device):
        nbytes = lib.gnnhwc_nchw_workspace_bytes(N, C, R, G, dt, 1)
        if nbytes == 0:
            raise RuntimeError("gnop::bwd_nchw: " + _cabi.last_error())
        stream = _current_stream_ptr(X.device)
        ws = _workspace(nbytes, X.device, stream)
        rc = lib.gnnhwc_bwd_nchw(
            dy.data_ptr(), X.data_ptr(), w_ptr, b_ptr,
            means.contiguous().data_ptr(), rstds.contiguous().data_ptr(),
            dX.data_ptr(), dweight.data_ptr() if dweight is not None else None, dbias.data_ptr() if dbias is not None else None,
            N, C, R, G, int(act_fn_option), dt, pdt, sdt,
            ws.data_ptr(), ws.numel(), stream)
    _cabi.check(rc, "gnop::bwd_nchw")
    return dX, dweight, dbias


def gn_nhwc_fwd_add(X, residual, channel_bias, weight, bias, G, eps, act_fn_option, return_sum):
    """gnop::fwd_add (no counterpart in the reference): gnop::fwd of S = X + residual + channel_bias[:, :, None],
    with the additions done inside the kernel.  X, residual: (N, C, R) channels-last views; channel_bias: (N, C).
    Returns (Y, S, means, rstds); S has no elements unless return_sum."""
    _check_device(X, "X")
    _check_device(weight, "weight")
    _check_device(bias, "bias")
    if X.dim() != 3:
        raise RuntimeError("gnop::fwd_add expects X of shape (N, C, R), got %s" % (tuple(X.shape),))
    N, C, R = X.shape
    dt = _dtype_code(X, "X")
    pdt = _dtype_code(weight, "weight")
    if bias.dtype != weight.dtype:
        raise RuntimeError("weight and bias must have the same dtype (%s vs %s)" % (weight.dtype, bias.dtype))
    if weight.numel() != C or bias.numel() != C:
        raise RuntimeError("weight and bias must have %d elements" % C)
    X_nrc = _as_nrc(X)
    res_ptr = cb_ptr = None
    cb_dt = dt
    if residual is not None:
        _check_device(residual, "residual")
        if residual.shape != X.shape or residual.dtype != X.dtype:
            raise RuntimeError("residual must have X's shape and dtype")
        res_nrc = _as_nrc(residual)
        res_ptr = res_nrc.data_ptr()
    if channel_bias is not None:
        _check_device(channel_bias, "channel_bias")
        if tuple(channel_bias.shape) != (N, C):
            raise RuntimeError("channel_bias must have shape (N, C) = (%d, %d)" % (N, C))
        cb_dt = _dtype_code(channel_bias, "channel_bias")
        channel_bias = channel_bias.contiguous()
        cb_ptr = channel_bias.data_ptr()
    Y = torch.empty_like(X_nrc)
    S = torch.empty_like(X_nrc) if return_sum else torch.empty((N, 0, C), dtype=X.dtype, device=X.device)
    sdtype = _stats_dtype(X.dtype)
    means = torch.empty((N, G), dtype=sdtype, device=X.device)
    rstds = torch.empty((N, G), dtype=sdtype, device=X.device)
    lib = _cabi.lib
    with _on_device(X.device):
        nbytes = lib.gnnhwc_fwd_workspace_bytes(N, R, C, G, dt)
        if nbytes == 0:
            raise RuntimeError("gnop::fwd_add: " + _cabi.last_error())
        stream = _current_stream_ptr(X.device)
        ws = _workspace(nbytes, X.device, stream)
        rc = lib.gnnhwc_fwd_add(
            X_nrc.data_ptr(), res_ptr, cb_ptr, S.data_ptr() if return_sum else None,
            weight.contiguous().data_ptr(), bias.contiguous().data_ptr(),
            Y.data_ptr(), means.data_ptr(), rstds.data_ptr(),
            N, R, C, G, float(eps), int(act_fn_option), dt, pdt, _DTYPE_CODE[sdtype], cb_dt,
            ws.data_ptr(), ws.numel(), stream)
    _cabi.check(rc, "gnop::fwd_add")
    return Y.permute(0, 2, 1), S.permute(0, 2, 1), means, rstds


# TORCH_LIBRARY(gnop, m) { m.def("fwd", ...); m.def("bwd", ...); } -- custom_gn.cpp:91-94.  The reference
# registers catch-all kernels that themselves reject non-device tensors; CompositeExplicitAutograd plays that
# role here, so a CPU tensor reaches the "must be a CUDA tensor" check instead of a dispatcher error.
_op_lib = torch.library.Library("gnop", "DEF")
_op_lib.define("fwd(Tensor X, Tensor weight, Tensor bias, int G, float eps, int act_fn_option) -> (Tensor, Tensor, Tensor)")
_op_lib.define("bwd(Tensor dy, Tensor X, Tensor weight, Tensor bias, Tensor means, Tensor rstds, int G, "
               "int act_fn_option) -> (Tensor, Tensor, Tensor)")
_op_lib.define("fwd_add(Tensor X, Tensor? residual, Tensor? channel_bias, Tensor weight, Tensor bias, int G, float eps, "
               "int act_fn_option, bool return_sum) -> (Tensor, Tensor, Tensor, Tensor)")
_op_lib.define("fwd_cast(Tensor X, Tensor? weight, Tensor? bias, int G, float eps, int act_fn_option, ScalarType out_dtype) -> "
               "(Tensor, Tensor, Tensor)")
_op_lib.define("fwd_nchw(Tensor X, Tensor weight, Tensor bias, int G, float eps, int act_fn_option) -> (Tensor, Tensor, Tensor)")
_op_lib.define("bwd_nchw(Tensor dy, Tensor X, Tensor weight, Tensor bias, Tensor means, Tensor rstds, int G, "
               "int act_fn_option) -> (Tensor, Tensor, Tensor)")
_op_lib.impl("fwd_nchw", gn_nchw_fwd, "CompositeExplicitAutograd")
_op_lib.impl("bwd_nchw", gn_nchw_bwd, "CompositeExplicitAutograd")
_op_lib.impl("fwd", gn_nhwc_fwd, "CompositeExplicitAutograd")
_op_lib.impl("fwd_cast", gn_nhwc_fwd_cast, "CompositeExplicitAutograd")
_op_lib.impl("fwd_add", gn_nhwc_fwd_add, "CompositeExplicitAutograd")
_op_lib.impl("bwd", gn_nhwc_bwd, "CompositeExplicitAutograd")


def _fwd_meta(X, weight, bias, G, eps, act_fn_option):
    """Shapes, dtypes and strides of gnop::fwd's outputs for meta / fake tensors (tracing): Y keeps X's
    (N, C, R) shape with strides (R*C, 1, C), as the permuted view returned by the real operator does."""
    N, C, R = X.shape
    Y = torch.empty((N, R, C), dtype=X.dtype, device=X.device).permute(0, 2, 1)
    sdtype = _stats_dtype(X.dtype)
    return Y, torch.empty((N, G), dtype=sdtype, device=X.device), torch.empty((N, G), dtype=sdtype, device=X.device)


def _bwd_meta(dy, X, weight, bias, means, rstds, G, act_fn_option):
    N, C, R = X.shape
    dX = torch.empty((N, R, C), dtype=X.dtype, device=X.device).permute(0, 2, 1)
    return dX, torch.empty((C,), dtype=weight.dtype, device=X.device), torch.empty((C,), dtype=weight.dtype, device=X.device)


def _fwd_add_meta(X, residual, channel_bias, weight, bias, G, eps, act_fn_option, return_sum):
    N, C, R = X.shape
    Y, means, rstds = _fwd_meta(X, weight, bias, G, eps, act_fn_option)
    S = torch.empty((N, R if return_sum else 0, C), dtype=X.dtype, device=X.device).permute(0, 2, 1)
    return Y, S, means, rstds


# The reference's operators cannot be traced (its forward is wrapped in torch._dynamo.disable, custom_gn.py:63);
# with these the operators carry correct output metadata under fake-tensor tracing.
_op_lib.impl("fwd", _fwd_meta, "Meta")
_op_lib.impl("bwd", _bwd_meta, "Meta")
_op_lib.impl("fwd_add", _fwd_add_meta, "Meta")


def _fwd_nchw_meta(X, weight, bias, G, eps, act_fn_option):
    N = X.shape[0]
    sdtype = _stats_dtype(X.dtype)
    return (torch.empty(X.shape, dtype=X.dtype, device=X.device), torch.empty((N, G), dtype=sdtype, device=X.device),
            torch.empty((N, G), dtype=sdtype, device=X.device))


def _bwd_nchw_meta(dy, X, weight, bias, means, rstds, G, act_fn_option):
    C = X.shape[1]
    return (torch.empty(X.shape, dtype=X.dtype, device=X.device), torch.empty((C,), dtype=weight.dtype, device=X.device),
            torch.empty((C,), dtype=weight.dtype, device=X.device))


_op_lib.impl("fwd_nchw", _fwd_nchw_meta, "Meta")
_op_lib.impl("bwd_nchw", _bwd_nchw_meta, "Meta")


def _fwd_setup_context(ctx, inputs, output):
    X, weight, bias, G, _eps, act_fn_option = inputs
    _Y, means, rstds = output
    ctx.save_for_backward(X, weight, bias, means, rstds)
    ctx.G = G
    ctx.act_fn_option = act_fn_option
    ctx.mark_non_differentiable(means, rstds)


def _fwd_backward(ctx, dY, _dmeans, _drstds):
    X, weight, bias, means, rstds = ctx.saved_tensors
    dY = dY.permute(0, 2, 1).contiguous().permute(0, 2, 1)  # X's own (R*C, 1, C) strides
    dX, dweight, dbias = torch.ops.gnop.bwd(dY, X, weight, bias, means, rstds, ctx.G, ctx.act_fn_option)
    return dX, dweight, dbias, None, None, None


# Autograd formula of gnop::fwd itself (the reference only differentiates through GN_NHWC_Func, custom_gn.py:29-47):
# with it and the meta kernels above, code that calls the operator directly can be traced and compiled whole.
torch.library.register_autograd("gnop::fwd", _fwd_backward, setup_context=_fwd_setup_context, lib=_op_lib)


def _fwd_cast_meta(X, weight, bias, G, eps, act_fn_option, out_dtype):
    N, C, R = X.shape
    Y = torch.empty((N, R, C), dtype=out_dtype, device=X.device).permute(0, 2, 1)
    sdtype = _stats_dtype(X.dtype)
    return Y, torch.empty((N, G), dtype=sdtype, device=X.device), torch.empty((N, G), dtype=sdtype, device=X.device)


_op_lib.impl("fwd_cast", _fwd_cast_meta, "Meta")


def _fwd_cast_setup_context(ctx, inputs, output):
    X, weight, bias, G, _eps, act_fn_option, _out_dtype = inputs
    _Y, means, rstds = output
    ctx.save_for_backward(X, weight, bias, means, rstds)
    ctx.G = G
    ctx.act_fn_option = act_fn_option
    ctx.mark_non_differentiable(means, rstds)


def _fwd_cast_backward(ctx, dY, _dmeans, _drstds):
    """The 16-bit gradient of Y goes to the backward kernels as it is (gnnhwc_bwd_cast widens it in registers)."""
    X, weight, bias, means, rstds = ctx.saved_tensors
    dY = dY.permute(0, 2, 1).contiguous().permute(0, 2, 1)
    if weight is None:
        dX, _dw, _db = gn_nhwc_bwd(dY, X, None, None, means, rstds, ctx.G, ctx.act_fn_option)
        return dX, None, None, None, None, None, None
    dX, dweight, dbias = torch.ops.gnop.bwd(dY, X, weight, bias, means, rstds, ctx.G, ctx.act_fn_option)
    return dX, dweight, dbias, None, None, None, None


torch.library.register_autograd("gnop::fwd_cast", _fwd_cast_backward, setup_context=_fwd_cast_setup_context, lib=_op_lib)


def _fwd_nchw_backward(ctx, dY, _dmeans, _drstds):
    X, weight, bias, means, rstds = ctx.saved_tensors
    dX, dweight, dbias = torch.ops.gnop.bwd_nchw(dY.contiguous(), X, weight, bias, means, rstds, ctx.G, ctx.act_fn_option)
    return dX, dweight, dbias, None, None, None


torch.library.register_autograd("gnop::fwd_nchw", _fwd_nchw_backward, setup_context=_fwd_setup_context, lib=_op_lib)


def _fwd_add_setup_context(ctx, inputs, output):
    X, residual, channel_bias, weight, bias, G, _eps, act_fn_option, return_sum = inputs
    _Y, S, means, rstds = output
    # the backward differentiates the normalisation at S: kept if it was materialised, else rebuilt from the inputs
    ctx.save_for_backward(S if return_sum else X, residual, channel_bias, weight, bias, means, rstds)
    ctx.have_sum = return_sum
    ctx.G = G
    ctx.act_fn_option = act_fn_option
    ctx.mark_non_differentiable(means, rstds)


def _fwd_add_backward(ctx, dY, dS, _dmeans, _drstds):
    first, residual, channel_bias, weight, bias, means, rstds = ctx.saved_tensors
    if ctx.have_sum:
        S = first
    else:
        acc = first.float() if first.dtype in (torch.float16, torch.bfloat16) else first
        if residual is not None:
            acc = acc + residual
        if channel_bias is not None:
            acc = acc + channel_bias.unsqueeze(-1)
        S = acc.to(first.dtype)
    S = S.permute(0, 2, 1).contiguous().permute(0, 2, 1)
    dY = dY.permute(0, 2, 1).contiguous().permute(0, 2, 1)
    dSum, dweight, dbias = torch.ops.gnop.bwd(dY, S, weight, bias, means, rstds, ctx.G, ctx.act_fn_option)
    if ctx.have_sum and dS is not None:
        dSum = dSum + dS
    dres = dSum if residual is not None else None
    dcb = None
    if channel_bias is not None:
        dcb = dSum.sum(dim=2, dtype=torch.float32).to(channel_bias.dtype)
    return dSum, dres, dcb, dweight, dbias, None, None, None, None


torch.library.register_autograd("gnop::fwd_add", _fwd_add_backward, setup_context=_fwd_add_setup_context, lib=_op_lib)


def group_norm_nhwc(x, weight, bias, num_groups, eps=1e-5, activation="identity", residual=None, channel_bias=None,
                    return_sum=False, out_dtype=None):
    """Functional, traceable form of GN_NHWC.forward for channels-last input (x.stride(1) == 1): the same operator
    and results, differentiated through the operator's registered autograd formula instead of GN_NHWC_Func, so
    torch.compile can keep it in one graph.  weight / bias must be given (use ones / zeros for a non-affine norm).

    Optional fused additions (no counterpart in the reference): the normalised tensor becomes
    s = x + residual + channel_bias[:, :, None, ...] (residual: x's shape; channel_bias: (N, C), e.g. a time
    embedding), computed inside the kernel and rounded to x's dtype once; with return_sum=True the call returns
    (y, s) so that s can serve as the next skip connection.

    out_dtype (no counterpart in the reference either): float32 input may leave as torch.float16 / torch.bfloat16,
    written in that type by the kernel (for a convolution that runs in half precision on a float32 residual stream);
    weight / bias may then be None.  Not combined with the fused additions."""
    if x.stride(1) != 1:
        raise RuntimeError("group_norm_nhwc expects channels-last input (stride 1 along dim 1)")
    if weight is not None and not torch.compiler.is_compiling():
        out = _native.group_norm(x, weight, bias, num_groups, eps, ACTIVATION_CODES[activation], out_dtype, residual, channel_bias,
                                 return_sum, True)
        if out is not NotImplemented:
            return out
    nd = x.dim()
    x = x.permute(0, *range(2, nd), 1).contiguous()  # (N, *spatial, C), a no-op copy-wise for channels-last input
    shape = x.shape
    R = 1
    for d in shape[1:-1]:
        R *= d
    X_flat = x.view(shape[0], R, shape[-1]).permute(0, 2, 1)
    code = ACTIVATION_CODES[activation]

    def unflat(t):
        return t.permute(0, 2, 1).reshape(shape).permute(0, nd - 1, *range(1, nd - 1))

    if out_dtype is not None and out_dtype != x.dtype:
        if residual is not None or channel_bias is not None or return_sum:
            raise RuntimeError("out_dtype cannot be combined with residual / channel_bias / return_sum")
        Y, _means, _rstds = torch.ops.gnop.fwd_cast(X_flat, weight, bias, num_groups, eps, code, out_dtype)
        return unflat(Y)
    if residual is None and channel_bias is None and not return_sum:
        Y, _means, _rstds = torch.ops.gnop.fwd(X_flat, weight, bias, num_groups, eps, code)
        return unflat(Y)
    R_flat = None
    if residual is not None:
        if residual.shape != torch.Size([shape[0], shape[-1], *shape[1:-1]]):
            raise RuntimeError("residual must have x's shape")
        R_flat = residual.permute(0, *range(2, nd), 1).contiguous().view(shape[0], R, shape[-1]).permute(0, 2, 1)
    Y, S, _means, _rstds = torch.ops.gnop.fwd_add(X_flat, R_flat, channel_bias, weight, bias, num_groups, eps, code, return_sum)
    return (unflat(Y), unflat(S)) if return_sum else unflat(Y)


class GN_NHWC_Func(torch.autograd.Function):
    """custom_gn.py:29-47.  apply(X, weight, bias, G, eps, activation_code) -> Y with X's shape and strides."""

    @staticmethod
    def forward(ctx, X, weight, bias, G, eps, activation):
        ctx.x_shape = X.shape
        R = 1
        for d in X.shape[2:]:
            R *= d
        X_flat = X.view(X.shape[0], X.shape[1], R)  # explicit R: "-1" is ambiguous for an empty batch
        # the operator's own implementation, called directly: going through torch.ops.gnop.fwd would add the
        # dispatcher and its autograd wrapper to every call, and this Function already is the autograd formula
        X_out, means, rstds = gn_nhwc_fwd(X_flat, weight, bias, G, eps, activation)
        ctx.save_for_backward(X_flat, weight, bias, means, rstds)
        ctx.G = G
        ctx.activation = activation
        return X_out.view(ctx.x_shape)

    @staticmethod
    def backward(ctx, dy):
        X_flat, weight, bias, means, rstds = ctx.saved_tensors
        # Bring dy into X's own layout (channels fastest, spatial dims in X's order).  The reference uses
        # dy.contiguous(memory_format=channels_last) (custom_gn.py:44), which only exists for 4-D tensors;
        # permuting the channel axis to the end and back works for any rank >= 3.
        nd = dy.dim()
        dy_last = dy.permute(0, *range(2, nd), 1).contiguous()
        dy_flat = dy_last.view(X_flat.shape[0], X_flat.shape[2], X_flat.shape[1]).permute(0, 2, 1)
        assert dy_flat.stride() == X_flat.stride() or X_flat.numel() == 0 or 1 in X_flat.shape
        dx, dgamma, dbeta = gn_nhwc_bwd(dy_flat, X_flat, weight, bias, means, rstds, ctx.G, ctx.activation)
        return dx.view(ctx.x_shape), dgamma, dbeta, None, None, None


class GN_NCHW_Func(torch.autograd.Function):
    """The same contract as GN_NHWC_Func for contiguous channels-first input (no counterpart in the reference,
    which lets torch handle that layout, custom_gn.py:75-79): apply(X, weight, bias, G, eps, activation_code) -> Y
    contiguous with X's shape."""

    @staticmethod
    def forward(ctx, X, weight, bias, G, eps, activation):
        ctx.x_shape = X.shape
        R = 1
        for d in X.shape[2:]:
            R *= d
        X_flat = X.contiguous().view(X.shape[0], X.shape[1], R)
        Y, means, rstds = gn_nchw_fwd(X_flat, weight, bias, G, eps, activation)
        ctx.save_for_backward(X_flat, weight, bias, means, rstds)
        ctx.G = G
        ctx.activation = activation
        return Y.view(ctx.x_shape)

    @staticmethod
    def backward(ctx, dy):
        X_flat, weight, bias, means, rstds = ctx.saved_tensors
        dy_flat = dy.contiguous().view(X_flat.shape)
        dx, dgamma, dbeta = gn_nchw_bwd(dy_flat, X_flat, weight, bias, means, rstds, ctx.G, ctx.activation)
        return dx.view(ctx.x_shape), dgamma, dbeta, None, None, None


_TORCH_ACTIVATIONS = (
    lambda t: t,
    F.relu,
    F.silu,
    F.gelu,
    lambda t: F.gelu(t, approximate="tanh"),
)


class GN_NHWC(nn.GroupNorm):
    """custom_gn.py:49-90.  GroupNorm over channels-last input with the activation applied in the same pass."""

    def __init__(self, num_groups, num_channels, activation="identity", out_dtype=None, **kwargs):
        super().__init__(num_groups, num_channels, **kwargs)
        self.activation = activation
        self.act_code = ACTIVATION_CODES[activation]  # unknown name -> KeyError, as in the reference
        # not in the reference: the type the result leaves in (None: the input's).  float32 channels-last device input
        # is written as float16 / bfloat16 by the kernel itself; any other combination is converted afterwards.
        self.out_dtype = out_dtype

    def forward(self, x):
        if not torch.compiler.is_compiling():
            # an ordinary eager call: checks, kernels and autograd node in native code (csrc/gn_torch.cpp), which declines
            # whatever it does not take -- the Python implementation below serves those calls, and their errors
            y = _native.group_norm(x, self.weight, self.bias, self.num_groups, self.eps, self.act_code, self.out_dtype, None, None,
                                   False)
            if y is not NotImplemented:
                return y
        if self.out_dtype is not None and self.out_dtype != x.dtype:
            if (x.is_cuda and x.dtype == torch.float32 and x.stride(1) == 1
                    and self.out_dtype in (torch.float16, torch.bfloat16)):
                return group_norm_nhwc(x, self.weight, self.bias, self.num_groups, self.eps, self.activation,
                                       out_dtype=self.out_dtype)
            return self._forward_same_dtype(x).to(self.out_dtype)
        return self._forward_same_dtype(x)

    def _forward_same_dtype(self, x):
        # The reference wraps this method in torch._dynamo.disable (custom_gn.py:63): its operators cannot be traced,
        # so a compiled model breaks its graph here.  These operators can (meta kernels + registered autograd), so
        # under torch.compile the same computation is expressed through them and stays inside the caller's graph.
        if torch.compiler.is_compiling():
            return self._forward_traced(x)
        if x.stride(1) == 1:
            # channels fastest.  Make the remaining dims contiguous in their logical order as well: a shape
            # (2, 3, 5, 9) input must have strides (135, 1, 27, 3), not e.g. (135, 1, 3, 15) (custom_gn.py:68-73).
            nd = x.dim()
            x = x.permute(0, *range(2, nd), 1).contiguous().permute(0, nd - 1, *range(1, nd - 1))
            run = GN_NHWC_Func.apply
        else:
            # channels-first input: the reference hands it to torch's GroupNorm and applies the activation in a
            # second pass (custom_gn.py:75-79); the same result (contiguous output) comes from the channels-first
            # kernels here, with the activation fused
            x = x.contiguous()
            if x.is_cuda:
                run = GN_NCHW_Func.apply
            else:
                # not a device tensor: exactly the reference's expression (its channels-first path never reaches a
                # kernel, so it also serves host tensors)
                act = _TORCH_ACTIVATIONS[self.act_code]

                def run(t, w, b, g, eps, _code):
                    return act(F.group_norm(t, g, w, b, eps))

        # affine=False: the reference materialises ones and zeros on every call (custom_gn.py:83-86); here the absent
        # parameters travel as None down to the kernels, which take NULL for gamma = 1, beta = 0
        return run(x, self.weight, self.bias, self.num_groups, self.eps, self.act_code)

    def _forward_traced(self, x):
        """forward() as torch.compile sees it: the same kernels through torch.ops.gnop.*, whose schemas take
        tensors only, so a normalisation without parameters passes ones and zeros here."""
        C = self.num_channels
        if self.affine:
            w, b = self.weight, self.bias
        else:
            w, b = x.new_ones((C,)), x.new_zeros((C,))
        if not x.is_cuda:
            return _TORCH_ACTIVATIONS[self.act_code](F.group_norm(x.contiguous(), self.num_groups, w, b, self.eps))
        if x.stride(1) == 1:
            return group_norm_nhwc(x, w, b, self.num_groups, self.eps, self.activation)
        shape = x.shape
        R = 1
        for d in shape[2:]:
            R *= d
        Y, _means, _rstds = torch.ops.gnop.fwd_nchw(x.contiguous().view(shape[0], C, R), w, b, self.num_groups, self.eps,
                                                    self.act_code)
        return Y.view(shape)

    def extra_repr(self):
        return "{num_groups}, {num_channels}, eps={eps}, affine={affine}, activation={activation}".format(**self.__dict__)
