"""Forward-only glue of a ConvNeXt-1D block on the GPU, one pass each, in place of the PyTorch
passes the reference spends around the operator (``models/convnext.py:306-318``: permute +
LayerNorm before the pointwise layers, layer scale + permute + residual after them; the
channels-last LayerNorm + GELU of the stem, ``:176-190``).  The harness uses them when no
gradient is being recorded; with autograd on it composes the same values from PyTorch ops."""
import ctypes

import torch
import torch.autograd.forward_ad as fwd
import torch.nn.functional as F

from . import _lib

_DTYPES = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}
MAX_C_ROWS, MAX_C_TILE = 2048, 1536


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _stream(t):
    return ctypes.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


def _f32(p):
    from .dwoconv1d import f32_copy
    return f32_copy(p)


def usable(x, C, tiled):
    """True when the fused kernels cover this call: CUDA tensor of a supported type, even C
    within the kernels' limit, and autograd switched off (they have no backward; with gradients
    enabled the callers compose the same values from PyTorch ops)."""
    return (x.is_cuda and x.dtype in _DTYPES and C % 2 == 0
            and C <= (MAX_C_TILE if tiled else MAX_C_ROWS) and not torch.is_grad_enabled())


def layernorm_nhwc(x, weight, bias, eps, gelu=False):
    """LayerNorm over the last dimension of a contiguous tensor (+ exact GELU)."""
    return _lib.host(x.get_device()).layernorm_nhwc(x, _f32(weight), _f32(bias), eps, gelu)


def nchw_layernorm_nhwc(x, weight, bias, eps):
    """[N,C,H,W] -> [N,H,W,C], LayerNorm over C: ``norm(x.permute(0, 2, 3, 1))`` in one pass."""
    return _lib.host(x.get_device()).nchw_layernorm_nhwc(x, _f32(weight), _f32(bias), eps)


def nhwc_scale_add_nchw(y, scale=None, residual=None):
    """[N,H,W,C] -> [N,C,H,W]: ``residual + (scale * y).permute(0, 3, 1, 2)`` in one pass
    (``scale`` [C] and ``residual`` [N,C,H,W] optional)."""
    sc = _f32(scale) if scale is not None else None
    return _lib.host(y.get_device()).nhwc_scale_add_nchw(y, sc, residual)


class _PointwiseLinear(torch.autograd.Function):
    """``F.linear`` whose parameter gradients come from the library: with a few input channels
    and every pixel of a batch as rows they are a reduction, not a matrix product."""

    @staticmethod
    def forward(ctx, x, w, b):
        ctx.set_materialize_grads(False)
        xc, wc, bc = x, w, b
        if torch.is_autocast_enabled(x.device.type):
            # the conversions of autocast, but not its own: gradients are off here, and the copies that
            # it keeps for the rest of the region would be cut off from the parameters
            dtype = torch.get_autocast_dtype(x.device.type)
            xc, wc, bc = (t if t is None else t.to(dtype) for t in (x, w, b))
        with torch.autocast(x.device.type, enabled=False):
            y = F.linear(xc, wc, bc)
        # (only what backward reads: parameters may be updated between the passes where the input takes
        # no gradient)
        ctx.save_for_backward(xc, w if ctx.needs_input_grad[0] else None)
        ctx.w_dtype, ctx.b_dtype = w.dtype, b.dtype if b is not None else None
        return y

    @staticmethod
    def backward(ctx, dy):
        if dy is None:
            return None, None, None
        x, w = ctx.saved_tensors
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            dx = torch.matmul(dy, w)
        need_db = ctx.b_dtype is not None and ctx.needs_input_grad[2]
        if ctx.needs_input_grad[1] or need_db:
            dy, x = dy.contiguous(), x.contiguous()
            if torch.is_grad_enabled() or dy.data_ptr() % 16 != 0 or dy.dtype != x.dtype:
                # gradients of gradients, or a piece of another buffer
                rows = dy.reshape(-1, dy.shape[-1])
                dw = torch.matmul(rows.t(), x.reshape(-1, x.shape[-1]).to(rows.dtype))
                db = rows.sum(0)
            else:
                dw, db = _lib.host(dy.get_device()).pointwise_wgrad(dy, x, need_db)
            dw = dw.to(ctx.w_dtype) if ctx.needs_input_grad[1] else None
            db = db.to(ctx.b_dtype) if need_db else None
        return dx, dw, db


def _eager(*tensors):
    """True for ordinary tensors in ordinary execution: no compilation, tracing, torch.func transform,
    dispatch mode, forward-mode derivative or tensor subclass, all of which an autograd function around native
    code would hide the layer from."""
    if (torch.compiler.is_compiling() or torch.jit.is_tracing()
            or torch._C._are_functorch_transforms_active() or torch._C._len_torch_dispatch_stack()):
        return False
    return all(t is None or (type(t) in (torch.Tensor, torch.nn.Parameter)
                             and fwd.unpack_dual(t).tangent is None) for t in tensors)


def pointwise_linear(x, linear):
    """``linear(x)`` of an ``nn.Linear`` with at most four inputs; where its parameters are being
    trained on a GPU, with the parameter gradients of ``dwo_pointwise_wgrad``."""
    w, b = linear.weight, linear.bias
    dtype = torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else x.dtype
    # (what autocast converts is saved converted, without its history: an input that is differentiated
    # itself stays with PyTorch then, whose gradients of gradients reach it and the weights)
    if (torch.is_grad_enabled() and _eager(x, w, b)
            and w.requires_grad and x.is_cuda and w.device == x.device and x.numel() > 0
            and (x.dtype == w.dtype == dtype or not x.requires_grad) and dtype in _DTYPES
            and all(t is None or t.dtype in _DTYPES for t in (x, w, b))
            and 1 <= x.shape[-1] <= 4
            and w.shape[0] * dtype.itemsize % 16 == 0 and w.shape[0] * dtype.itemsize <= 4096):
        return _PointwiseLinear.apply(x, w, b)
    return F.linear(x, w, b)


def pointwise_dwconv_nhwc(x, linear, conv):
    """``conv(linear(x))`` for a channels-last ``x`` [N,H,W,Cin] (Cin <= 4), an ``nn.Linear``
    Cin -> C and an NHWC ``DepthwiseOrientedConv1d`` over C channels, without writing the
    C-channel tensor (the stem's ``dw1(pw1(x))``, models/convnext.py:177-178)."""
    if not x.is_cuda or x.dtype not in _DTYPES:
        raise RuntimeError("x must be a CUDA tensor of type float32, bfloat16 or float16")
    x = x.contiguous()
    N, H, W, Cin = x.shape
    C, K, stride = conv.out_channels, conv.kernel_size[1], conv.stride[0]
    w = _f32(conv.weight)
    if conv.resid is not None:
        w = w + conv.resid.to(w)
    taps, layouts = conv._taps.lookup(conv.theta, C, K, x.device)  # cached per theta version
    P, Q = -(-H // stride), -(-W // stride)
    y = torch.empty((N, P, Q, C), dtype=x.dtype, device=x.device)
    pw_w = _f32(linear.weight)
    pw_b = _f32(linear.bias) if linear.bias is not None else None
    w2 = w.reshape(C, K)
    cb = _f32(conv.bias) if conv.bias is not None else None
    _lib.check(_lib.ready(x.device).dwo_pointwise_fprop(
        _ptr(x), _ptr(pw_w), _ptr(pw_b), _ptr(w2), _ptr(cb), _ptr(taps), _ptr(y), N, Cin, C, H, W,
        K, stride, _DTYPES[x.dtype], layouts[x.element_size()], _stream(x)), "dwo_pointwise_fprop")
    return y
