"""Glue of a ConvNeXt-1D block on the GPU, one pass each, in place of the PyTorch passes the
reference spends around the operator (``models/convnext.py:306-318``: permute + LayerNorm before the
pointwise layers, layer scale + permute + residual after them; the channels-last LayerNorm + GELU
of the stem, ``:176-190``).  The first functions are forward only, for calls under ``no_grad``; the
autograd functions below them are what a training pass runs, for ordinary tensors and modules (no
transforms, tracing, subclasses or hooks: those compose the same values from PyTorch ops)."""
import ctypes

import torch
import torch.nn.functional as F
import torch.nn.modules.module as _mod

from . import _lib
from .dwoconv1d import DepthwiseOrientedConv1d, KernelTuple, _native_covers, f32_copy as _f32, ordinary

_DTYPES = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}
MAX_C_ROWS, MAX_C_TILE = 2048, 1536
MAX_C_TRAIN = 1024


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _stream(t):
    return ctypes.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


def usable(x, C, tiled):
    """True when the fused kernels cover this call: CUDA tensor of a supported type, even C
    within the kernels' limit, and autograd switched off (they have no backward; with gradients
    enabled the callers compose the same values from PyTorch ops)."""
    return (x.is_cuda and x.dtype in _DTYPES and C % 2 == 0
            and C <= (MAX_C_TILE if tiled else MAX_C_ROWS) and not torch.is_grad_enabled())


def _pieces(x, C):
    """True where the kernels that take eight channels per lane cover LayerNorm over C channels of x."""
    return x.is_cuda and x.dtype in _DTYPES and C % 8 == 0 and 8 <= C <= MAX_C_TRAIN and 0 < x.numel() < 1 << 31


def layernorm_nhwc(x, weight, bias, eps, gelu=False):
    """LayerNorm over the last dimension of a contiguous tensor (+ exact GELU)."""
    host, C = _lib.host(x.get_device()), x.shape[-1]
    if _pieces(x, C):
        return host.ln_rows(x, _f32(weight), _f32(bias), eps, gelu, x.dtype, False)[0]
    return host.layernorm_nhwc(x, _f32(weight), _f32(bias), eps, gelu)


def nchw_layernorm_nhwc(x, weight, bias, eps):
    """[N,C,H,W] -> [N,H,W,C], LayerNorm over C: ``norm(x.permute(0, 2, 3, 1))`` in one pass."""
    host = _lib.host(x.get_device())
    if x.dim() == 4 and _pieces(x, x.shape[1]):
        return host.ln_tile(x, _f32(weight), _f32(bias), eps, False, x.dtype, False)[0]
    return host.nchw_layernorm_nhwc(x, _f32(weight), _f32(bias), eps)


def nhwc_scale_add_nchw(y, scale=None, residual=None):
    """[N,H,W,C] -> [N,C,H,W]: ``residual + (scale * y).permute(0, 3, 1, 2)`` in one pass
    (``scale`` [C] and ``residual`` [N,C,H,W] optional)."""
    sc = _f32(scale) if scale is not None else None
    return _lib.host(y.get_device()).nhwc_scale_add_nchw(y, sc, residual)


# A product kernel's launch, a workgroup of 256 threads per 128 rows and 96 or 128 outputs, has fewer than 2^32 threads below so many
# inputs (eight per row at least; more than 2^37 outputs do not fit the card)
_PRODUCT_MAX = 1 << 33


def _layer16(x, w, b):
    """True where the product kernels of the library cover ``F.linear(x, w, b)`` without gradients: 16-bit tensors of one type on
    one GPU, sizes in multiples of eight."""
    return (not torch.is_grad_enabled() and x.is_cuda and x.numel() > 0 and x.dtype in (torch.bfloat16, torch.float16)
            and w.dtype == x.dtype and w.device == x.device and w.shape[1] == x.shape[-1]
            and (b is None or (b.dtype == x.dtype and b.device == x.device))
            and w.shape[0] % 8 == 0 and w.shape[1] % 8 == 0 and max(w.shape) <= 65536 and ordinary(x, w, b)
            and not torch.is_autocast_enabled(x.device.type) and x.numel() < _PRODUCT_MAX)


def linear_gelu(x, linear):
    """``F.gelu(linear(x))``; without gradients one kernel where the library covers it."""
    w, b = linear.weight, linear.bias
    if plain(linear, Linear) and x.dim() >= 2 and _layer16(x, w, b):
        return _lib.host(x.get_device()).linear_rows(x, w, b, True)
    return F.gelu(linear(x))


# Above this many inputs and rows the library's product and a pass for the tail are faster than linear_planes, which
# stages both operands through 64 columns at a time (25088 x 768 x 3072 in bf16: 49 against 61 us; 1568 rows 30 against 29; 25088 x
# 384 x 1536 57 against 58)
_PLANES_MAX_K, _PLANES_MAX_ROWS = 2048, 2048


def linear_tail(x, linear, gamma, residual):
    """``residual + (gamma * linear(x)).permute(0, 3, 1, 2)`` without gradients; gamma may be None."""
    w, b = linear.weight, linear.bias
    if (plain(linear, Linear) and x.dim() == 4 and _layer16(x, w, b) and residual.dtype == x.dtype
            and (gamma is None or (gamma.dtype == x.dtype and gamma.device == x.device))
            and (w.shape[1] <= _PLANES_MAX_K or x.numel() // w.shape[1] <= _PLANES_MAX_ROWS)):
        return _lib.host(x.get_device()).linear_planes(x, w, b, gamma, residual)
    return nhwc_scale_add_nchw(linear(x), gamma, residual)


def norm_planes(x, before, linear, norm):
    """``norm(linear(F.gelu(before(x)))).permute(0, 3, 1, 2)`` without gradients as one kernel where the library covers it (the stem's
    64 inputs, 96 or 128 outputs), else None."""
    w, b = linear.weight, linear.bias
    if not (plain(linear, Linear) and x.dim() == 4 and w.shape[1] == 64 and w.shape[0] in (96, 128) and _layer16(x, w, b)
            and x.numel() < 1 << 37):
        return None
    affine = before.weight, before.bias, norm.weight, norm.bias
    if any(p is None or p.device != x.device or p.shape != (C,) for p, C in zip(affine, (64, 64, w.shape[0], w.shape[0]))):
        return None
    g0, b0, g1, b1 = map(_f32, affine)
    return _lib.host(x.get_device()).linear_norm_planes(x, g0, b0, before.eps, w, b, g1, b1, norm.eps)


# Rows from which both layers run as one kernel: enough workgroups of 128 pixels that its long chain is paid for (bf16, us, behind a
# pass over other memory, two kernels / one: 10240 x 96 16.1 / 17.8, 12288 x 96 18.4 / 18.0; 16384 x 128 20.9 / 25.3, 16640 x 128, where the
# first product has more tiles than the chip holds, 30.8 / 25.4; 25088 x 192 44.3 / 43.9, 29008 x 192 47.7 / 45.0, in odd planes 29008 68 /
# 75, 34300 99 / 90).  There is no instance for 256 channels.
_MLP_ROWS = {96: 12288, 128: 16385, 192: 28672, 384: 21846}
# At 384 channels a workgroup has a CU to itself (101 KB of LDS): its time goes in rounds of 256 workgroups, about 100 us each, and
# the last round pays from two thirds on (20384 rows 82 / 101, 21952 112 / 102, 32732 148 / 112, 32928 151 / 199, 39200 171 / 199, 43120 201 /
# 202, 49000 218 / 206, 65660 313 / 308; back to back the second round from three quarters on, 43904 181 / 199, 50960 216 / 197)
_MLP_ROUND = 32768


def _mlp_pays(C, rows):
    """True where ``block_mlp`` is the faster route for this many rows of C channels."""
    return rows >= _MLP_ROWS.get(C, rows + 1) and (C != 384 or 3 * rows >= 2 * _MLP_ROUND * -(-rows // _MLP_ROUND))


def block_mlp(y, first, second, gamma, residual):
    """``linear_tail(linear_gelu(y, first), second, gamma, residual)`` as one kernel where that is faster, else None."""
    C = y.shape[-1]
    if not _mlp_pays(C, y.numel() // max(C, 1)):
        return None
    w1, b1, w2, b2 = first.weight, first.bias, second.weight, second.bias
    if not (y.dim() == 4 and plain(first, Linear)
            and plain(second, Linear) and b1 is not None and b2 is not None and w1.shape == (4 * C, C)
            and w2.shape == (C, 4 * C) and _layer16(y, w1, b1) and residual.dtype == y.dtype
            and all(t is None or (t.dtype == y.dtype and t.device == y.device) for t in (w2, b2, gamma))
            and ordinary(w2, b2, gamma, residual)):
        return None
    return _lib.host(y.get_device()).block_mlp(y, w1, b1, w2, b2, gamma, residual)


def infer_block(x, block, conv, inner):
    """A ConvNeXt-1D block (operator ``conv``) or 1D++ block (and ``inner``, between the pointwise layers) without gradients: the
    kernels of its layers one by one, with what they check checked once for all of them (layer by layer 45 to 50 us of host time
    per block, four launches of which are 19); None where one of them would not take the path that is taken here."""
    if (torch.compiler.is_compiling() or torch.is_grad_enabled() or not x.is_cuda or x.dim() != 4 or x.numel() == 0
            or x.dtype not in (torch.bfloat16, torch.float16) or torch.is_autocast_enabled("cuda")):
        return None
    layers = block._modules
    first, last, norm = layers.get("pwconv1"), layers.get("pwconv2"), layers.get("norm")
    if not (plain(conv, DepthwiseOrientedConv1d) and plain(first, Linear) and plain(last, Linear)
            and type(norm) is torch.nn.LayerNorm and (inner is None or plain(inner, DepthwiseOrientedConv1d))):
        return None
    N, C, H, W = x.shape
    rows, dtype, device = N * H * W, x.dtype, x.device
    p, q, r, s = conv._parameters, first._parameters, last._parameters, norm._parameters
    w, theta, g, b = p.get("weight"), p.get("theta"), s.get("weight"), s.get("bias")
    w1, b1, w2, b2 = q.get("weight"), q.get("bias"), r.get("weight"), r.get("bias")
    bias, gamma = conv.bias, block.gamma
    module = conv.module_fp32_large if conv.arbitrary_size else conv.module_fp32
    if (w is None or theta is None or g is None or b is None or w1 is None or b1 is None or w2 is None or b2 is None
            or conv.nhwc or conv.resid is not None or type(module) is not KernelTuple or module.stride != 1
            or C % 8 != 0 or C > MAX_C_TILE
            or 4 * rows * C >= _PRODUCT_MAX or w1.shape != (4 * C, C) or w2.shape != (C, 4 * C)
            or not _native_covers(x, w, theta, bias, None, module, False) or not ordinary(g, b, w1, b1, w2, b2, gamma)):
        return None
    for t in (w1, b1, w2, b2) if gamma is None else (w1, b1, w2, b2, gamma):
        if t.dtype != dtype or t.device != device:
            return None
    if g.device != device or b.device != device:
        return None
    if inner is not None:
        v, angles, vb, resid = inner._parameters.get("weight"), inner._parameters.get("theta"), inner.bias, inner.resid
        wide = inner.module_fp32_large if inner.arbitrary_size else inner.module_fp32
        if not (v is not None and angles is not None and inner.nhwc and type(wide) is KernelTuple and wide.stride == 1
                and v.shape[0] == 4 * C and v.shape[-1] == wide.kernel_size and v.is_floating_point()
                and ordinary(v, angles, vb, resid) and all(t is None or t.device == device for t in (v, vb, resid))):
            return None
        taps, layouts = wide.taps.lookup(angles, 4 * C, v.shape[-1], device)
    host, x = _lib.host(x.get_device()), x.contiguous()
    y = host.conv_norm(x, _f32(w), None if bias is None else _f32(bias),
                       module.taps.lookup(theta, C, w.shape[-1], device)[0], _f32(g), _f32(b), norm.eps, _pieces(x, C))
    if inner is None and _mlp_pays(C, rows):
        return host.block_mlp(y, w1, b1, w2, b2, gamma, x)
    y = host.linear_rows(y, w1, b1, True)
    if inner is not None:
        v = _f32(v)
        y = host.fprop(y, v if resid is None else v + resid.to(v), taps, 1, None if vb is None else _f32(vb),
                       layouts[x.element_size()])
    if 4 * C <= _PLANES_MAX_K or rows <= _PLANES_MAX_ROWS:
        return host.linear_planes(y, w2, b2, gamma, x)
    return host.nhwc_scale_add_nchw(F.linear(y, w2, b2), None if gamma is None else _f32(gamma), x)


class _PointwiseLinear(torch.autograd.Function):
    """``F.linear`` in the library: with a few input channels and every pixel of a batch as rows it is a pass over its output,
    and its parameter gradients are a reduction, not matrix products."""

    @staticmethod
    def forward(ctx, x, w, b):
        ctx.set_materialize_grads(False)
        xc, wc, bc = x, w, b
        if torch.is_autocast_enabled(x.device.type):
            # the conversions of autocast, but not its own: gradients are off here, and the copies that
            # it keeps for the rest of the region would be cut off from the parameters
            dtype = torch.get_autocast_dtype(x.device.type)
            xc, wc, bc = (t if t is None else t.to(dtype) for t in (x, w, b))
        if xc.dtype != torch.float32 and wc.shape[0] % 64 == 0:
            y = _lib.host(xc.get_device()).pointwise_forward(xc, wc, bc)
        else:
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


def pointwise_linear(x, linear):
    """``linear(x)`` of an ``nn.Linear`` with at most four inputs; where its parameters are being
    trained on a GPU, with the parameter gradients of ``dwo_pointwise_wgrad``."""
    w, b = linear.weight, linear.bias
    dtype = torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else x.dtype
    # (what autocast converts is saved converted, without its history: an input that is differentiated
    # itself stays with PyTorch then, whose gradients of gradients reach it and the weights)
    if (torch.is_grad_enabled() and ordinary(x, w, b)
            and w.requires_grad and x.is_cuda and w.device == x.device and x.numel() > 0
            and (x.dtype == w.dtype == dtype or not x.requires_grad) and dtype in _DTYPES
            and all(t is None or t.dtype in _DTYPES for t in (x, w, b))
            and 1 <= x.shape[-1] <= 4
            and w.shape[0] * dtype.itemsize % 16 == 0 and w.shape[0] * dtype.itemsize <= 4096):
        return _PointwiseLinear.apply(x, w, b)
    return F.linear(x, w, b)


def plain(module, *types):
    """True where calling the module is calling its class's own forward: no subclass, no hooks."""
    return (type(module) in types and not (module._forward_hooks or module._forward_pre_hooks
                                           or module._backward_hooks or module._backward_pre_hooks)
            and not (_mod._global_forward_hooks or _mod._global_forward_pre_hooks
                     or _mod._global_backward_hooks or _mod._global_backward_pre_hooks)
            and "forward" not in module.__dict__)


def _recording(*tensors):
    """True where the training kernels may stand for a composition of PyTorch ops on these tensors (None for
    an absent one): gradients are being recorded, on one GPU, for ordinary non-empty tensors of a known type."""
    x = tensors[0]
    return (torch.is_grad_enabled() and x.is_cuda and x.numel() > 0 and ordinary(*tensors)
            and all(t is None or (t.device == x.device and t.dtype in _DTYPES) for t in tensors))


def _autocast(x):
    """The type that autocast converts a pointwise layer's tensors to here, or None."""
    return torch.get_autocast_dtype(x.device.type) if torch.is_autocast_enabled(x.device.type) else None


def _norm_type(x, C, norm, consumer):
    """Output type of LayerNorm over C channels of x: fp32 under autocast, or what autocast makes of it for ``consumer``
    where nothing but that plain pointwise layer sees it; None where the kernels do not cover the call."""
    w, b = norm.weight, norm.bias
    if w is None or b is None or w.shape != (C,) or b.shape != (C,) or C % 8 != 0 or C > MAX_C_TRAIN:
        return None
    ac = _autocast(x)
    if ac is None:
        return x.dtype if x.dtype == w.dtype == b.dtype else None
    out = ac if ac in _DTYPES and consumer is not None and plain(consumer, Linear) else torch.float32
    return out if x.dtype == out or torch.float32 in (x.dtype, out) else None


def _second_order(value, inputs, needed, dout):
    """Gradients of ``value(*inputs)`` with their own history (a backward pass that is being recorded), for the inputs that
    ``needed`` marks: what was saved has to be what ``apply`` was given, a copy made inside ``forward`` has no history."""
    leaves = [t for t, n in zip(inputs, needed) if n]
    with torch.autocast(dout.device.type, enabled=False):
        y = value(*inputs)
        got = iter(torch.autograd.grad(y, leaves, dout, create_graph=True, allow_unused=True))
    return [next(got) if n else None for n in needed]


def _patches(x):
    """[N,H,W,C] -> [N,H/2,W/2,4C]: the 2 x 2 patches, channel first (an odd last row or column is in none)."""
    N, H, W, C = x.shape
    x = x[:, :H // 2 * 2, :W // 2 * 2].reshape(N, H // 2, 2, W // 2, 2, C)
    return x.permute(0, 1, 3, 5, 2, 4).reshape(N, H // 2, W // 2, 4 * C)


class _TileNorm(torch.autograd.Function):
    """LayerNorm over dim 1 of an NCHW tensor, as [N,H,W,C] or as 2 x 2 patches."""

    @staticmethod
    def forward(ctx, x, w, b, eps, dtype, patches=False):
        ctx.set_materialize_grads(False)
        out, stats = _lib.host(x.get_device()).ln_tile(x, _f32(w), _f32(b), eps, patches, dtype, True)
        ctx.save_for_backward(x, w, b, stats)
        ctx.eps, ctx.dtype, ctx.patches = eps, dtype, patches
        return out

    @staticmethod
    def backward(ctx, dout):
        if dout is None:
            return None, None, None, None, None, None
        x, w, b, stats = ctx.saved_tensors
        if torch.is_grad_enabled():
            def value(x, w, b):
                y = F.layer_norm(x.permute(0, 2, 3, 1).float(), w.shape, w.float(), b.float(), ctx.eps)
                return (_patches(y) if ctx.patches else y).to(ctx.dtype)
            return (*_second_order(value, (x, w, b), ctx.needs_input_grad[:3], dout), None, None, None)
        dx, dw, db = _lib.host(x.get_device()).ln_tile_backward(dout, x, stats, _f32(w), ctx.patches, w.dtype)
        return dx, dw, db.to(b.dtype), None, None, None


class _RowNorm(torch.autograd.Function):
    """LayerNorm over the last dimension (gelu & 1: + exact GELU, gelu & 2: of the value rounded to the output's type)."""

    @staticmethod
    def forward(ctx, x, w, b, eps, gelu, dtype):
        ctx.set_materialize_grads(False)
        out, stats = _lib.host(x.get_device()).ln_rows(x, _f32(w), _f32(b), eps, gelu, dtype, True)
        ctx.save_for_backward(x, w, b, stats)
        ctx.eps, ctx.gelu, ctx.dtype = eps, gelu, dtype
        return out

    @staticmethod
    def backward(ctx, dout):
        if dout is None:
            return None, None, None, None, None, None
        x, w, b, stats = ctx.saved_tensors
        if torch.is_grad_enabled():
            def value(x, w, b):
                y = F.layer_norm(x.float(), w.shape, w.float(), b.float(), ctx.eps)
                if ctx.gelu & 2:
                    y = y.to(ctx.dtype).float()
                return (F.gelu(y) if ctx.gelu else y).to(ctx.dtype)
            return (*_second_order(value, (x, w, b), ctx.needs_input_grad[:3], dout), None, None, None)
        dx, dw, db = _lib.host(x.get_device()).ln_rows_backward(dout, x, stats, _f32(w), _f32(b), ctx.gelu, w.dtype)
        return dx, dw, db.to(b.dtype), None, None, None


class _BlockTail(torch.autograd.Function):
    """``x + (gamma * y).permute(0, 3, 1, 2)`` in ``dtype`` for y [N,H,W,C] and x [N,C,H,W] (``rounded``: the product is a
    tensor of y's type by itself); without gamma and x the permutation alone."""

    @staticmethod
    def forward(ctx, y, gamma, x, dtype, rounded):
        ctx.set_materialize_grads(False)
        out = _lib.host(y.get_device()).block_tail(y, None if gamma is None else _f32(gamma), x, dtype, rounded)
        ctx.save_for_backward(*(() if gamma is None else (y, gamma)))
        ctx.types = y.dtype, None if x is None else x.dtype
        return out

    @staticmethod
    def backward(ctx, dout):
        if dout is None:
            return None, None, None, None, None
        dtype, x_dtype = ctx.types
        dx = dout.to(x_dtype) if ctx.needs_input_grad[2] else None
        if not (ctx.needs_input_grad[0] or ctx.needs_input_grad[1]):
            return None, None, dx, None, None
        y, gamma = ctx.saved_tensors or (None, None)  # (read once: hooks, as of checkpointing, may unpack a tensor only once)
        if torch.is_grad_enabled():
            if gamma is None:
                return dout.permute(0, 2, 3, 1).to(dtype), None, dx, None, None

            def value(y, gamma):
                return (gamma * y).permute(0, 3, 1, 2).to(dout.dtype)
            return (*_second_order(value, (y, gamma), ctx.needs_input_grad[:2], dout), dx, None, None)
        scale, grad = (None, torch.float32) if gamma is None else (_f32(gamma), gamma.dtype)
        dy, dg = _lib.host(dout.get_device()).block_tail_backward(dout, y, scale, dtype, grad)
        return dy, dg, dx, None, None


class _Linear(torch.autograd.Function):
    """``F.linear`` over 16-bit activations whose parameter gradients come from ``dwo_linear_wgrad``, in the parameters'
    own type.  ``wc`` is w in x's type where w has another one: an input of its own, so that the copy of the forward pass is
    what the backward pass reads, with its history where that pass is recorded; w takes the whole gradient otherwise."""

    @staticmethod
    def forward(ctx, x, w, wc, b):
        ctx.set_materialize_grads(False)
        wc = w if wc is None else wc
        y = F.linear(x, wc, b if b is None else b.to(x.dtype))
        # (only what backward reads: parameters may be updated between the passes where the input takes no gradient, and
        # always where they were converted)
        ctx.save_for_backward(x, wc if ctx.needs_input_grad[0] else None)
        ctx.w_dtype, ctx.b_dtype = w.dtype, b.dtype if b is not None else None
        return y

    @staticmethod
    def backward(ctx, dy):
        if dy is None:
            return None, None, None, None
        x, wc = ctx.saved_tensors
        dx = dw = db = None
        need_db = ctx.b_dtype is not None and ctx.needs_input_grad[3]
        if ctx.needs_input_grad[0]:
            dx = torch.matmul(dy, wc)
        if torch.is_grad_enabled():  # gradients of gradients: with the history of x and of the weights
            rows = dy.reshape(-1, dy.shape[-1])
            if ctx.needs_input_grad[1]:
                dw = torch.matmul(rows.t(), x.reshape(-1, x.shape[-1])).to(ctx.w_dtype)
            if need_db:
                db = rows.sum(0).to(ctx.b_dtype)
            return dx, dw, None, db
        if ctx.needs_input_grad[1] or need_db:
            dw, db = _lib.host(x.get_device()).linear_wgrad(dy, x, need_db, ctx.w_dtype)
            if need_db and ctx.b_dtype != ctx.w_dtype:
                db = db.to(ctx.b_dtype)
        return dx, dw if ctx.needs_input_grad[1] else None, None, db


def _linear16(x, w, b):
    """``F.linear(x, w, b)`` for a 16-bit x and parameters of any type.  (Conversions as autocast makes them, recorded, but
    not kept for the rest of its region.)"""
    return _Linear.apply(x, w, None if w.dtype == x.dtype else w.to(x.dtype), b)


class Linear(torch.nn.Linear):
    """``nn.Linear``; where it is trained over 16-bit activations on a GPU, its parameter gradients are one pass
    over them (``dwo_linear_wgrad``)."""

    def forward(self, x):
        w, b = self.weight, self.bias
        if (w.requires_grad and w.shape[0] % 8 == 0 and w.shape[1] % 8 == 0 and max(w.shape) <= 65536
                and x.dim() >= 1 and x.shape[-1] == w.shape[1] and _recording(x, w, b)
                and x.numel() // w.shape[1] <= 1 << 31 and w.numel() + w.shape[0] < 1 << 31):  # (two threads per gradient)
            ac = _autocast(x)
            dtype = ac or x.dtype
            if dtype in (torch.bfloat16, torch.float16) and (
                    ac is not None or (x.dtype == w.dtype and (b is None or b.dtype == w.dtype))):
                return _linear16(x.to(dtype), w, b)
        return F.linear(x, w, b)


def tile_norm(x, norm, consumer=None):
    """LayerNorm (the parameters and eps of ``norm``) over dim 1 of an NCHW tensor as [N,H,W,C], recorded by autograd, in
    the type that ``consumer`` (the pointwise layer that alone reads it) takes; None where the kernels do not cover the
    call."""
    if not (_recording(x, norm.weight, norm.bias) and x.dim() == 4 and x.numel() < 1 << 31):
        return None
    dtype = _norm_type(x, x.shape[1], norm, consumer)
    return None if dtype is None else _TileNorm.apply(x.contiguous(), norm.weight, norm.bias, norm.eps, dtype)


def row_norm(x, norm, gelu=False, consumer=None):
    """``norm(x)`` of an ``nn.LayerNorm`` over the last dimension (then exact GELU), as ``tile_norm``."""
    if not (_recording(x, norm.weight, norm.bias) and plain(norm, torch.nn.LayerNorm) and x.dim() >= 2
            and x.numel() // max(x.shape[-1], 1) < 1 << 31):
        return None
    dtype = _norm_type(x, x.shape[-1], norm, consumer)
    # (without autocast a 16-bit LayerNorm's output is a 16-bit tensor by itself)
    mode = 0 if not gelu else 1 if _autocast(x) is not None or dtype == torch.float32 else 3
    return None if dtype is None else _RowNorm.apply(x.contiguous(), norm.weight, norm.bias, norm.eps, mode, dtype)


def _tail_covers(y):
    if y.dim() != 4 or y.shape[-1] % 8 != 0 or y.shape[-1] > MAX_C_TRAIN or y.numel() >= 1 << 31:
        return False
    N, H, W, C = y.shape  # (fewer than 2^32 threads: 256 per 64 pixels x 64 channels of an image)
    return N * -(-H * W // 64) * -(-C // 64) < 1 << 24


def block_tail(y, gamma, x):
    """``x + (gamma * y).permute(0, 3, 1, 2)`` recorded by autograd; None where the kernels do not cover the call."""
    if not (_recording(y, gamma, x) and _tail_covers(y) and gamma.shape == y.shape[-1:]
            and x.shape == (y.shape[0], y.shape[3], y.shape[1], y.shape[2])):
        return None
    dtype = torch.promote_types(torch.promote_types(gamma.dtype, y.dtype), x.dtype)
    if dtype not in (y.dtype, torch.float32) or x.dtype not in (y.dtype, dtype):
        return None
    product = torch.promote_types(gamma.dtype, y.dtype)
    return _BlockTail.apply(y.contiguous(), gamma, x, dtype, product == y.dtype != torch.float32)


def planes(y):
    """``y.permute(0, 3, 1, 2).contiguous()``, recorded by autograd where the kernels cover it."""
    if _recording(y) and _tail_covers(y):
        return _BlockTail.apply(y.contiguous(), None, None, y.dtype, False)
    return y.permute(0, 3, 1, 2).contiguous()


def downsample(x, norm, conv):
    """``conv(norm(x))`` of a LayerNorm over the channels of an NCHW tensor and a 2 x 2 convolution of stride 2: a pointwise layer
    over normalised patches, with the weights as they lie in memory.  None where the kernels do not cover the call."""
    w, b = conv.weight, conv.bias
    if not (plain(conv, torch.nn.Conv2d) and conv.kernel_size == (2, 2) == conv.stride and conv.padding == (0, 0)
            and conv.dilation == (1, 1) and conv.groups == 1 and conv.padding_mode == "zeros"
            and x.dim() == 4 and x.is_cuda and min(x.shape[2:]) >= 2 and 0 < x.numel() < 1 << 31
            and w.shape[1] == x.shape[1] and w.shape[0] % 8 == 0 and x.shape[1] % 8 == 0 and x.shape[1] <= MAX_C_TRAIN
            and w.shape[0] <= MAX_C_TRAIN and w.is_contiguous()
            and norm.weight.shape == norm.bias.shape == x.shape[1:2]):
        return None
    rows = w.view(w.shape[0], -1)
    if torch.is_grad_enabled():
        if not (_recording(x, norm.weight, norm.bias, w, b) and w.requires_grad):
            return None
        ac = _autocast(x)
        dtype = ac or x.dtype
        if dtype not in (torch.bfloat16, torch.float16) or x.dtype not in (dtype, torch.float32):
            return None
        if ac is None and not (x.dtype == norm.weight.dtype == norm.bias.dtype == w.dtype
                               and (b is None or b.dtype == w.dtype)):
            return None
        p = _TileNorm.apply(x.contiguous(), norm.weight, norm.bias, norm.eps, dtype, True)
        return planes(_linear16(p, rows, b))
    if norm.weight.device != x.device or not _layer16(x.permute(0, 2, 3, 1), w[:, :, 0, 0], b) or not ordinary(w):
        return None
    host = _lib.host(x.get_device())
    p = host.ln_tile(x, _f32(norm.weight), _f32(norm.bias), norm.eps, True, x.dtype, False)[0]
    return host.linear_planes(p, rows, b, None, None)


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
